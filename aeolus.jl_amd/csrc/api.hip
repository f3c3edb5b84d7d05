// The C ABI of libaeolus_hip (declared in include/aeolus_hip.h).
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "../../include/aeolus_hip.h"
#include "kernels.h"

using namespace aeo;

namespace {

thread_local char g_err[1024] = "";

int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

#define HIPCHK(x)                                                                              \
    do {                                                                                       \
        hipError_t e_ = (x);                                                                   \
        if (e_ != hipSuccess) return fail(AEO_ERR_HIP, "%s: %s", #x, hipGetErrorString(e_));   \
    } while (0)

struct Context {
    int device = -1;
    hipStream_t stream = nullptr;
    bool profile = false;
    struct Rec {
        std::vector<std::pair<hipEvent_t, hipEvent_t>> ev;
        int count = 0;
        double ms = 0;
    };
    std::map<std::string, Rec> prof;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> pool;
    double *red = nullptr;  // device scratch of the reductions read back by the host
    size_t red_n = 0;
};
Context *g_ctx = nullptr;

// At least n doubles of the context's reduction scratch (grown, never shrunk).
// Every user launches into it and reads the result back (synchronising the
// stream) before it returns, so consecutive calls on the stream may share it.
static double *red_scratch(size_t n) {
    if (g_ctx->red_n < n) {
        if (g_ctx->red) {
            hipStreamSynchronize(g_ctx->stream);
            hipFree(g_ctx->red);
        }
        g_ctx->red = nullptr;
        g_ctx->red_n = 0;
        if (hipMalloc(&g_ctx->red, sizeof(double) * n) != hipSuccess) return nullptr;
        g_ctx->red_n = n;
    }
    return g_ctx->red;
}

// timing of one launch site: events recorded on the library stream
struct Timed {
    Context::Rec *rec = nullptr;
    hipEvent_t b{}, e{};
    Timed(const char *name) {
        if (!g_ctx || !g_ctx->profile) return;
        rec = &g_ctx->prof[name];
        if (!g_ctx->pool.empty()) {
            b = g_ctx->pool.back().first;
            e = g_ctx->pool.back().second;
            g_ctx->pool.pop_back();
        } else {
            hipEventCreate(&b);
            hipEventCreate(&e);
        }
        hipEventRecord(b, g_ctx->stream);
    }
    ~Timed() {
        if (!rec) return;
        hipEventRecord(e, g_ctx->stream);
        rec->ev.push_back({b, e});
    }
};

void profile_collect() {
    if (!g_ctx) return;
    bool any = false;
    for (auto &kv : g_ctx->prof) any |= !kv.second.ev.empty();
    if (!any) return;
    hipStreamSynchronize(g_ctx->stream);
    for (auto &kv : g_ctx->prof) {
        for (auto &p : kv.second.ev) {
            float ms = 0;
            hipEventElapsedTime(&ms, p.first, p.second);
            kv.second.ms += ms;
            kv.second.count++;
            g_ctx->pool.push_back(p);
        }
        kv.second.ev.clear();
    }
}

#define NEED_CTX() \
    if (!g_ctx) return fail(AEO_ERR_STATE, "aeo_init has not been called")

}  // namespace

aeo::ProfScope::ProfScope(const char *name) {
    if (name && g_ctx && g_ctx->profile) impl = new Timed(name);
}
aeo::ProfScope::~ProfScope() { delete (Timed *)impl; }

// ---------------------------------------------------------------------------
// grid
// ---------------------------------------------------------------------------
struct aeo_grid {
    int Nx, Ny, Nz, H;
    double dx, dy, dz;
    int stretched;
    std::vector<double> idzc, idzf, wlo, whi, alo, ahi;  // host, storage levels
    std::vector<double> dzc, dzf;                         // host, storage levels (Nz+2H, Nz+2H+1)
    double *d64[6] = {};                                 // device copies
    float *d32[6] = {};
    Metrics<double> m64;
    Metrics<float> m32;
};

template <typename T> static const Metrics<T> &metrics(const aeo_grid *g);
template <> const Metrics<double> &metrics<double>(const aeo_grid *g) { return g->m64; }
template <> const Metrics<float> &metrics<float>(const aeo_grid *g) { return g->m32; }

template <typename T>
static void fill_metrics(Metrics<T> &m, const aeo_grid *g, T *const *dv) {
    m.Nx = g->Nx; m.Ny = g->Ny; m.Nz = g->Nz; m.H = g->H;
    m.sx = g->Nx + 2 * g->H; m.sy = g->Ny + 2 * g->H; m.sz = g->Nz + 2 * g->H;
    m.idx = T(1 / g->dx); m.idy = T(1 / g->dy);
    m.idx2 = T(1 / (g->dx * g->dx)); m.idy2 = T(1 / (g->dy * g->dy));
    m.stretched = g->stretched;
    m.idz = T(1 / g->dz); m.idz2 = T(1 / (g->dz * g->dz));
    m.teno_ct = T(1e-5);  // TENO(N; C_T = 1e-5), src/AdvectionSchemes.jl:535
    m.idzc = dv[0]; m.idzf = dv[1]; m.wlo = dv[2]; m.whi = dv[3]; m.alo = dv[4]; m.ahi = dv[5];
}

extern "C" int aeo_grid_create(int Nx, int Ny, int Nz, int H, double dx, double dy, double dz,
                               const double *zf_interior, aeo_grid **out) {
    NEED_CTX();
    if (!out) return fail(AEO_ERR_ARG, "aeo_grid_create: null output handle");
    if (Nx < 1 || Ny < 1 || Nz < 1) return fail(AEO_ERR_ARG, "size must be positive, got (%d,%d,%d)", Nx, Ny, Nz);
    if (H < 1) return fail(AEO_ERR_ARG, "halo must be >= 1, got %d", H);
    if (Nx < H || Ny < H || Nz <= H) return fail(AEO_ERR_ARG, "interior (%d,%d,%d) must exceed the halo %d", Nx, Ny, Nz, H);
    if (!(dx > 0) || !(dy > 0)) return fail(AEO_ERR_ARG, "dx, dy must be positive");
    // the kernels address storage arrays with 32-bit offsets
    if ((double)(Nx + 2 * H) * (Ny + 2 * H) * (Nz + 2 * H) * 8.0 >= 2147483648.0)
        return fail(AEO_ERR_UNSUPPORTED, "storage (%d+2H)(%d+2H)(%d+2H) exceeds 2 GiB per FP64 array", Nx, Ny, Nz);
    auto g = std::make_unique<aeo_grid>();
    g->Nx = Nx; g->Ny = Ny; g->Nz = Nz; g->H = H; g->dx = dx; g->dy = dy; g->dz = dz;
    const int n = Nz + 2 * H;
    g->idzc.assign(n, 0); g->idzf.assign(n + 1, 0);
    g->wlo.assign(n, 0); g->whi.assign(n, 0); g->alo.assign(n, 0); g->ahi.assign(n, 0);
    if (!zf_interior) {
        if (!(dz > 0)) return fail(AEO_ERR_ARG, "dz must be positive");
        g->stretched = 0;
        for (int k = 0; k < n; k++) g->idzc[k] = 1 / dz;
        for (int k = 0; k <= n; k++) g->idzf[k] = 1 / dz;
        g->dzc.assign(n, dz);
        g->dzf.assign(n + 1, dz);
    } else {
        g->stretched = 1;
        for (int k = 0; k < Nz; k++)
            if (!(zf_interior[k + 1] > zf_interior[k]))
                return fail(AEO_ERR_ARG, "custom face vector must be strictly increasing");
        // _extend_faces, src/StretchedGrids.jl:319-337 (1-based k -> 0-based k-1)
        std::vector<double> zf(n + 1), zc(n), dzc(n), dzf(n + 1);
        for (int k = 1; k <= Nz + 1; k++) zf[H + k - 1] = zf_interior[k - 1];
        for (int k = H; k >= 1; k--) zf[k - 1] = 2 * zf[k] - zf[k + 1];
        for (int k = H + Nz + 2; k <= n + 1; k++) zf[k - 1] = 2 * zf[k - 2] - zf[k - 3];
        // StretchedGrid constructor, :375-388
        for (int k = 0; k < n; k++) dzc[k] = zf[k + 1] - zf[k];
        for (int k = 0; k < n; k++) zc[k] = (zf[k] + zf[k + 1]) / 2;
        dzf[0] = dzc[0];
        for (int k = 1; k < n; k++) dzf[k] = zc[k] - zc[k - 1];
        dzf[n] = dzc[n - 1];
        g->dzc = dzc;
        g->dzf = dzf;
        // level_metrics, :570-600
        for (int k = 0; k < n; k++) g->idzc[k] = 1 / dzc[k];
        for (int k = 0; k <= n; k++) g->idzf[k] = 1 / dzf[k];
        for (int k = 1; k < n; k++) {
            g->wlo[k] = dzc[k] / (dzc[k - 1] + dzc[k]);
            g->whi[k] = dzc[k - 1] / (dzc[k - 1] + dzc[k]);
            double s = dzc[k - 1] + dzc[k];
            g->alo[k] = dzc[k - 1] / s;
            g->ahi[k] = dzc[k] / s;
        }
    }
    const std::vector<double> *vs[6] = {&g->idzc, &g->idzf, &g->wlo, &g->whi, &g->alo, &g->ahi};
    for (int q = 0; q < 6; q++) {
        size_t len = vs[q]->size();
        HIPCHK(hipMalloc(&g->d64[q], sizeof(double) * len));
        HIPCHK(upload_dev(g->d64[q], vs[q]->data(), sizeof(double) * len));
        std::vector<float> f(len);
        for (size_t c = 0; c < len; c++) f[c] = (float)(*vs[q])[c];
        HIPCHK(hipMalloc(&g->d32[q], sizeof(float) * len));
        HIPCHK(upload_dev(g->d32[q], f.data(), sizeof(float) * len));
    }
    fill_metrics<double>(g->m64, g.get(), g->d64);
    fill_metrics<float>(g->m32, g.get(), g->d32);
    *out = g.release();
    return AEO_OK;
}

extern "C" int aeo_grid_destroy(aeo_grid *g) {
    if (!g) return AEO_OK;
    for (int q = 0; q < 6; q++) {
        hipFree(g->d64[q]);
        hipFree(g->d32[q]);
    }
    delete g;
    return AEO_OK;
}

extern "C" int aeo_grid_metrics(const aeo_grid *g, double *idzc, double *idzf) {
    if (!g) return fail(AEO_ERR_ARG, "null grid");
    if (idzc) memcpy(idzc, g->idzc.data(), sizeof(double) * g->idzc.size());
    if (idzf) memcpy(idzf, g->idzf.data(), sizeof(double) * g->idzf.size());
    return AEO_OK;
}

// ---------------------------------------------------------------------------
// context and memory
// ---------------------------------------------------------------------------
extern "C" const char *aeo_last_error(void) { return g_err; }

// What built the library: compiler, HIP version, target (the build half of
// provenance(), src/io/run_folder.jl:215-260)
extern "C" const char *aeo_build_info(void) {
#define AEO_STR2(x) #x
#define AEO_STR(x) AEO_STR2(x)
    return "libaeolus_hip; compiler: " __clang_version__ "; HIP " AEO_STR(HIP_VERSION_MAJOR) "." AEO_STR(
        HIP_VERSION_MINOR) "." AEO_STR(HIP_VERSION_PATCH) "; target gfx950; built " __DATE__ " " __TIME__;
#undef AEO_STR
#undef AEO_STR2
}

// The device a run used: name, gfx architecture, compute units, HBM bytes
extern "C" int aeo_device_info(int device, char *name, size_t name_len, char *arch, size_t arch_len, int *cus,
                               size_t *mem_bytes) {
    if (!name || !arch || !cus || !mem_bytes || name_len == 0 || arch_len == 0)
        return fail(AEO_ERR_ARG, "null argument");
    hipDeviceProp_t pr;
    HIPCHK(hipGetDeviceProperties(&pr, device));
    snprintf(name, name_len, "%s", pr.name);
    snprintf(arch, arch_len, "%s", pr.gcnArchName);
    *cus = pr.multiProcessorCount;
    *mem_bytes = pr.totalGlobalMem;
    return AEO_OK;
}

extern "C" int aeo_init(int device) {
    if (g_ctx) {
        if (g_ctx->device == device) return AEO_OK;
        return fail(AEO_ERR_STATE, "already initialised on device %d", g_ctx->device);
    }
    int n = 0;
    HIPCHK(hipGetDeviceCount(&n));
    if (device < 0 || device >= n) return fail(AEO_ERR_ARG, "device %d out of range (%d devices)", device, n);
    HIPCHK(hipSetDevice(device));
    auto c = std::make_unique<Context>();
    c->device = device;
    HIPCHK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    // the device address of the allocation-free entry point's scratch, once per device
    if (device < NOALLOC_MAX_DEVICES) {
        const hipError_t e = noalloc_bind(device);
        if (e != hipSuccess) {
            hipStreamDestroy(c->stream);
            return fail(AEO_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        }
    }
    g_ctx = c.release();
    return AEO_OK;
}

extern "C" int aeo_shutdown(void) {
    if (!g_ctx) return AEO_OK;
    hipStreamSynchronize(g_ctx->stream);
    for (auto &kv : g_ctx->prof)
        for (auto &p : kv.second.ev) g_ctx->pool.push_back(p);
    for (auto &p : g_ctx->pool) {
        hipEventDestroy(p.first);
        hipEventDestroy(p.second);
    }
    hipStreamDestroy(g_ctx->stream);
    if (g_ctx->red) hipFree(g_ctx->red);
    delete g_ctx;
    g_ctx = nullptr;
    return AEO_OK;
}

extern "C" int aeo_sync(void) {
    NEED_CTX();
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_malloc(void **dptr, size_t bytes) {
    NEED_CTX();
    if (!dptr) return fail(AEO_ERR_ARG, "null pointer");
    HIPCHK(hipMalloc(dptr, bytes ? bytes : 1));
    return AEO_OK;
}
extern "C" int aeo_free(void *dptr) {
    NEED_CTX();
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    HIPCHK(hipFree(dptr));
    return AEO_OK;
}
extern "C" int aeo_memcpy_h2d(void *dst, const void *src, size_t bytes) {
    NEED_CTX();
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_ctx->stream));
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    return AEO_OK;
}
extern "C" int aeo_memcpy_d2h(void *dst, const void *src, size_t bytes) {
    NEED_CTX();
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_ctx->stream));
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    return AEO_OK;
}
__global__ void copy_kernel(uint4 *__restrict__ dst, const uint4 *__restrict__ src, size_t n) {
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x)
        dst[t] = src[t];
}

// the STREAM triad a = b + s·c over n doubles, 8-byte accesses (the width of
// the solver's vector kernels): the bandwidth reference (reads 16n bytes,
// writes 8n) and the calibration dispatch of the HBM traffic counters
// (one element per work item in 1024-wide groups: the fastest of the
// launch shapes measured on MI355X, ≈ 6.1 TB/s at 1 GiB per array)
__global__ void __launch_bounds__(1024) triad_kernel(double *__restrict__ a, const double *__restrict__ b,
                                                     const double *__restrict__ c, double s, size_t n) {
    const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (t < n) a[t] = b[t] + s * c[t];
}

extern "C" int aeo_stream_triad(double *a, const double *b, const double *c, double s, long long n) {
    NEED_CTX();
    if (!a || !b || !c || n < 0) return fail(AEO_ERR_ARG, "null argument or negative size");
    Timed t("triad");
    if (n == 0) return AEO_OK;
    const size_t nb = ((size_t)n + 1023) / 1024;
    if (nb > 0x7fffffffULL) return fail(AEO_ERR_ARG, "triad: n too large");
    hipLaunchKernelGGL(triad_kernel, dim3((unsigned)nb), dim3(1024), 0, g_ctx->stream, a, b, c, s, (size_t)n);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_memcpy_d2d(void *dst, const void *src, size_t bytes) {
    NEED_CTX();
    if (!dst || !src) return fail(AEO_ERR_ARG, "null argument");
    Timed t("copy");
    if (bytes % 16 || ((uintptr_t)dst | (uintptr_t)src) % 16) {
        // sizes or pointers off the 16-byte grid: the runtime's copy, same stream
        HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, g_ctx->stream));
        return AEO_OK;
    }
    size_t n = bytes / 16;
    hipLaunchKernelGGL(copy_kernel, dim3(4096), dim3(256), 0, g_ctx->stream, (uint4 *)dst, (const uint4 *)src, n);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_memset(void *dptr, int value, size_t bytes) {
    NEED_CTX();
    HIPCHK(hipMemsetAsync(dptr, value, bytes, g_ctx->stream));
    return AEO_OK;
}

// ---------------------------------------------------------------------------
// halos and advection
// ---------------------------------------------------------------------------
static int check_bc(int bc) { return bc == AEO_PERIODIC || bc == AEO_NOFLUX || bc == AEO_WALL; }

extern "C" int aeo_fill_halos(aeo_grid *g, int precision, void *field, int loc, int bc_x, int bc_y, int bc_z) {
    NEED_CTX();
    if (!g || !field) return fail(AEO_ERR_ARG, "null argument");
    if (!check_bc(bc_x) || !check_bc(bc_y) || !check_bc(bc_z) || loc < 0 || loc > 3)
        return fail(AEO_ERR_ARG, "bad location or boundary kind");
    if (bc_x == AEO_WALL || bc_y == AEO_WALL)
        return fail(AEO_ERR_UNSUPPORTED, "ImpermeableWall is a z boundary (the reference fills walls in z only)");
    Timed t("halo");
    if (precision == AEO_F64) launch_halo<double>(g_ctx->stream, (double *)field, g->Nx, g->Ny, g->Nz, g->H, loc, bc_x, bc_y, bc_z);
    else if (precision == AEO_F32) launch_halo<float>(g_ctx->stream, (float *)field, g->Nx, g->Ny, g->Nz, g->H, loc, bc_x, bc_y, bc_z);
    else return fail(AEO_ERR_ARG, "bad precision %d", precision);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

static int required_halo(int scheme) {
    switch (scheme) {
    case AEO_CENTERED: case AEO_UPWIND: return 1;
    case AEO_WENO5: case AEO_WENO_JS5: case AEO_WENO_Z5: return 3;
    case AEO_WENO_Z7: return 4;
    case AEO_TENO5: return 3;
    case AEO_TENO8: return 5;  // required_halo(::TENO{8}), src/AdvectionSchemes.jl:569
    case AEO_VARIANCE_CONSERVING: return 1;
    }
    return -1;
}

// the schemes of the momentum operator and of the step: the reconstructions
// the fused kernels are built for (TENO and the skew form are scalar operators)
static int check_step_scheme(int scheme) {
    if (scheme == AEO_TENO5 || scheme == AEO_TENO8 || scheme == AEO_VARIANCE_CONSERVING)
        return fail(AEO_ERR_UNSUPPORTED, "scheme %d is a scalar advection operator here; momentum and the step take "
                                         "centered, upwind, weno5, weno_js5, weno_z5 or weno_z7", scheme);
    return AEO_OK;
}

static int check_scheme(const aeo_grid *g, int scheme, int p) {
    int h = required_halo(scheme);
    if (h < 0) return fail(AEO_ERR_ARG, "unknown advection scheme %d", scheme);
    if ((scheme == AEO_WENO_Z5 || scheme == AEO_WENO_Z7) && p != 1 && p != 2)
        return fail(AEO_ERR_ARG, "WENO-Z τ-exponent p must be 1 or 2 (got %d)", p);
    // _check_halo, src/AdvectionSchemes.jl:668-674; the momentum stencils read
    // one more cell across for the transporting velocity
    if (g->H < h) return fail(AEO_ERR_ARG, "scheme %d advection requires halo >= %d (got %d)", scheme, h, g->H);
    if (g->H < 2) return fail(AEO_ERR_ARG, "this build needs halo >= 2");
    return AEO_OK;
}

static int advect_scalar_ct(aeo_grid *g, int precision, int scheme, int p, double C_T, void *tend, const void *u,
                            const void *v, const void *w, const void *phi) {
    NEED_CTX();
    if (!g || !tend || !u || !v || !w || !phi) return fail(AEO_ERR_ARG, "null argument");
    int rc = check_scheme(g, scheme, p);
    if (rc) return rc;
    Timed t("advect");
    if (scheme == AEO_VARIANCE_CONSERVING) {
        // _advect_variance_conserving! has a RegularGrid method only (:1440-1446)
        if (g->stretched) return fail(AEO_ERR_UNSUPPORTED, "advect_variance_conserving!: regular grids");
        if (precision == AEO_F64)
            launch_varcons<double>(g_ctx->stream, g->m64, (double *)tend, (const double *)u, (const double *)v,
                                   (const double *)w, (const double *)phi);
        else if (precision == AEO_F32)
            launch_varcons<float>(g_ctx->stream, g->m32, (float *)tend, (const float *)u, (const float *)v,
                                  (const float *)w, (const float *)phi);
        else return fail(AEO_ERR_ARG, "bad precision %d", precision);
        HIPCHK(hipGetLastError());
        return AEO_OK;
    }
    if (precision == AEO_F64) {
        Metrics<double> m = g->m64;
        m.teno_ct = C_T;
        rc = launch_advect<double>(g_ctx->stream, m, 0, scheme, p, (const double *)u, (const double *)v,
                                   (const double *)w, (const double *)phi, nullptr, nullptr, nullptr, (double *)tend);
    } else if (precision == AEO_F32) {
        Metrics<float> m = g->m32;
        m.teno_ct = (float)C_T;
        rc = launch_advect<float>(g_ctx->stream, m, 0, scheme, p, (const float *)u, (const float *)v,
                                  (const float *)w, (const float *)phi, nullptr, nullptr, nullptr, (float *)tend);
    } else return fail(AEO_ERR_ARG, "bad precision %d", precision);
    if (rc) return fail(AEO_ERR_ARG, "advection launch failed");
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_advect_scalar(aeo_grid *g, int precision, int scheme, int p, void *tend, const void *u,
                                 const void *v, const void *w, const void *phi) {
    return advect_scalar_ct(g, precision, scheme, p, 1e-5, tend, u, v, w, phi);
}

// advect_teno!(tend, u, v, w, ϕ; order, C_T, q) (src/AdvectionSchemes.jl:750-756)
extern "C" int aeo_advect_teno(aeo_grid *g, int precision, int order, double C_T, int q, void *tend, const void *u,
                               const void *v, const void *w, const void *phi) {
    if (order != 5 && order != 8) return fail(AEO_ERR_ARG, "TENO order must be 5 or 8 (got %d)", order);
    if (!(C_T > 0)) return fail(AEO_ERR_ARG, "TENO cut-off C_T must be positive (got %g)", C_T);
    if (q != 6) return fail(AEO_ERR_UNSUPPORTED, "this build's TENO uses the exponent q = 6 (got %d)", q);
    return advect_scalar_ct(g, precision, order == 5 ? AEO_TENO5 : AEO_TENO8, 2, C_T, tend, u, v, w, phi);
}

// FluxLimiterWorkspace(mesh) (src/AdvectionSchemes.jl:800-822). The
// reference keeps the face fluxes F and L and the ratio R; the two tiled
// passes here recompute F and L where they are used, so the workspace is
// the ratio R alone, one storage-sized array of the grid at one precision
struct aeo_flux_workspace {
    const aeo_grid *g;
    int precision;
    void *ratio;
};

extern "C" int aeo_flux_limiter_workspace_create(aeo_grid *g, int precision, aeo_flux_workspace **out) {
    NEED_CTX();
    if (!g || !out) return fail(AEO_ERR_ARG, "null argument");
    if (precision != AEO_F64 && precision != AEO_F32) return fail(AEO_ERR_ARG, "bad precision %d", precision);
    auto *ws = new aeo_flux_workspace{g, precision, nullptr};
    const size_t bytes = (size_t)(g->Nx + 2 * g->H) * (g->Ny + 2 * g->H) * (g->Nz + 2 * g->H) *
                         (precision == AEO_F64 ? 8 : 4);
    if (hipMalloc(&ws->ratio, bytes) != hipSuccess || zero_dev(ws->ratio, bytes) != hipSuccess) {
        if (ws->ratio) hipFree(ws->ratio);
        delete ws;
        return fail(AEO_ERR_HIP, "flux limiter workspace: out of device memory");
    }
    *out = ws;
    return AEO_OK;
}

extern "C" int aeo_flux_limiter_workspace_destroy(aeo_flux_workspace *ws) {
    if (!ws) return AEO_OK;
    if (g_ctx) hipStreamSynchronize(g_ctx->stream);
    if (ws->ratio) hipFree(ws->ratio);
    delete ws;
    return AEO_OK;
}

// advect_positive!(tend, u, v, w, ϕ, dt; scheme, p, workspace, bcs, accumulate)
// (src/AdvectionSchemes.jl:1135-1160)
extern "C" int aeo_advect_positive(aeo_grid *g, int precision, int scheme, int p, double C_T, void *tend,
                                   const void *u, const void *v, const void *w, const void *phi, double dt,
                                   aeo_flux_workspace *ws, const int *bcs, int accumulate) {
    NEED_CTX();
    if (!g || !tend || !u || !v || !w || !phi) return fail(AEO_ERR_ARG, "null argument");
    if (precision != AEO_F64 && precision != AEO_F32) return fail(AEO_ERR_ARG, "bad precision %d", precision);
    // _reconstruction (:1692-1702): :weno5 names WENO-JS5 on this path; no :upwind
    if (scheme == AEO_WENO5) scheme = AEO_WENO_JS5;
    if (scheme != AEO_CENTERED && scheme != AEO_WENO_JS5 && scheme != AEO_WENO_Z5 && scheme != AEO_WENO_Z7 &&
        scheme != AEO_TENO5 && scheme != AEO_TENO8)
        return fail(AEO_ERR_ARG, "advect_positive!: unknown reconstruction %d; expected centered, weno5, "
                                 "weno_js5, weno_z5, weno_z7, teno5 or teno8", scheme);
    if ((scheme == AEO_TENO5 || scheme == AEO_TENO8) && !(C_T > 0))
        return fail(AEO_ERR_ARG, "TENO cut-off C_T must be positive (got %g)", C_T);
    int rc = check_scheme(g, scheme, p);
    if (rc) return rc;
    // _check_stretched_recon (:839-843)
    if (g->stretched && scheme != AEO_CENTERED)
        return fail(AEO_ERR_ARG, "advect_positive! on a StretchedGrid takes scheme = :centered only (the stencil "
                                 "assumes uniform spacing)");
    if (bcs)
        for (int q = 0; q < 3; q++)
            if (bcs[q] < AEO_PERIODIC || bcs[q] > AEO_WALL) return fail(AEO_ERR_ARG, "bad boundary condition");
    if (ws && (ws->g != g || ws->precision != precision))
        return fail(AEO_ERR_ARG, "the flux limiter workspace belongs to another grid or precision");
    aeo_flux_workspace *own = nullptr;
    if (!ws) {  // the reference allocates a workspace per call when none is passed
        rc = aeo_flux_limiter_workspace_create(g, precision, &own);
        if (rc) return rc;
        ws = own;
    }
    Timed t("advect_positive");
    Metrics<double> m64 = g->m64;
    Metrics<float> m32 = g->m32;
    m64.teno_ct = C_T;
    m32.teno_ct = (float)C_T;
    if (precision == AEO_F64) {
        rc = launch_advect_positive<double>(g_ctx->stream, m64, scheme, p, (double *)tend, (const double *)u,
                                            (const double *)v, (const double *)w, (const double *)phi, dt,
                                            (double *)ws->ratio, bcs, accumulate);
    } else {
        rc = launch_advect_positive<float>(g_ctx->stream, m32, scheme, p, (float *)tend, (const float *)u,
                                           (const float *)v, (const float *)w, (const float *)phi, (float)dt,
                                           (float *)ws->ratio, bcs, accumulate);
    }
    const hipError_t e = hipGetLastError();
    if (own) aeo_flux_limiter_workspace_destroy(own);
    if (rc) return fail(AEO_ERR_ARG, "advect_positive launch failed");
    HIPCHK(e);
    return AEO_OK;
}

extern "C" int aeo_advect_momentum(aeo_grid *g, int precision, int scheme, int p, void *tu, void *tv, void *tw,
                                   const void *u, const void *v, const void *w) {
    NEED_CTX();
    if (!g || !tu || !tv || !tw || !u || !v || !w) return fail(AEO_ERR_ARG, "null argument");
    int rc = check_step_scheme(scheme);
    if (rc) return rc;
    rc = check_scheme(g, scheme, p);
    if (rc) return rc;
    Timed t("advect");
    if (precision == AEO_F64)
        rc = launch_advect<double>(g_ctx->stream, g->m64, 1, scheme, p, (const double *)u, (const double *)v,
                                   (const double *)w, nullptr, (double *)tu, (double *)tv, (double *)tw, nullptr);
    else if (precision == AEO_F32)
        rc = launch_advect<float>(g_ctx->stream, g->m32, 1, scheme, p, (const float *)u, (const float *)v,
                                  (const float *)w, nullptr, (float *)tu, (float *)tv, (float *)tw, nullptr);
    else return fail(AEO_ERR_ARG, "bad precision %d", precision);
    if (rc) return fail(AEO_ERR_ARG, "advection launch failed");
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

// ---------------------------------------------------------------------------
// pressure solvers
// ---------------------------------------------------------------------------
struct aeo_unet;
struct aeo_poisson {
    int kind = 0;  // 0 fft, 1 column, 2 MG-preconditioned CG, 3 multigrid cycles, 4 flexible CG (learned)
    int Nx, Ny, Nz;
    bool periodic_x, periodic_y, periodic_z;
    SpectralPlan *sp = nullptr;
    MGPlan *mg = nullptr;
    double tol = 0;
    int maxit = 0;
    double *src = nullptr, *phi = nullptr;  // interior-sized FP64
    int iters = 0, status = AEO_DIRECT;
    double resid = NAN;
    // flexible CG: the multigrid solver whose operator and V-cycle it uses
    aeo_poisson *base = nullptr;
    aeo_unet *net = nullptr;
    const double *mask = nullptr;
    int mode = 0, use_guess = 0;
    FCGState *fcg = nullptr;
};

static int poisson_alloc(aeo_poisson *h) {
    size_t n = (size_t)h->Nx * h->Ny * h->Nz;
    HIPCHK(hipMalloc(&h->src, sizeof(double) * n));
    HIPCHK(hipMalloc(&h->phi, sizeof(double) * n));
    HIPCHK(hipMemsetAsync(h->src, 0, sizeof(double) * n, g_ctx->stream));
    HIPCHK(hipMemsetAsync(h->phi, 0, sizeof(double) * n, g_ctx->stream));
    return AEO_OK;
}

extern "C" int aeo_poisson_fft_create(int Nx, int Ny, int Nz, double dx, double dy, double dz, aeo_poisson **out) {
    NEED_CTX();
    if (!out) return fail(AEO_ERR_ARG, "null output handle");
    auto h = std::make_unique<aeo_poisson>();
    h->kind = 0; h->Nx = Nx; h->Ny = Ny; h->Nz = Nz;
    h->periodic_x = h->periodic_y = h->periodic_z = true;
    char err[512] = "";
    h->sp = spectral_create(Nx, Ny, Nz, g_ctx->stream, err, sizeof err);
    if (!h->sp) return fail(AEO_ERR_UNSUPPORTED, "%s", err);
    int rc = spectral_fft_setup(h->sp, dx, dy, dz);
    if (rc == -2) { spectral_destroy(h->sp); return fail(AEO_ERR_UNSUPPORTED, "FFT solver: Nz (%d) must be a product of 2, 3 and 5 in 2..512", Nz); }
    if (rc) { spectral_destroy(h->sp); return fail(AEO_ERR_HIP, "FFT solver setup failed"); }
    rc = poisson_alloc(h.get());
    if (rc) return rc;
    *out = h.release();
    return AEO_OK;
}

extern "C" int aeo_poisson_column_create(int Nx, int Ny, int Nz, double dx, double dy, int bc_x, int bc_y,
                                         const double *lower, const double *upper, const double *hweight,
                                         const double *measure, const double *inv_coupling, const double *gauge,
                                         aeo_poisson **out) {
    NEED_CTX();
    if (!out || !lower || !upper || !hweight || !measure || !inv_coupling || !gauge)
        return fail(AEO_ERR_ARG, "null argument");
    // src/PressureSolvers.jl:631-636
    if (!(lower[0] == 0 && upper[Nz - 1] == 0))
        return fail(AEO_ERR_ARG, "the bottom and top faces carry no flux: lower[1] = upper[Nz] = 0");
    for (int bc : {bc_x, bc_y})
        if (bc != AEO_PERIODIC && bc != AEO_NOFLUX)
            return fail(AEO_ERR_ARG, "column solver: lateral boundaries periodic (R2HC) or Neumann (REDFT10)");
    auto h = std::make_unique<aeo_poisson>();
    h->kind = 1; h->Nx = Nx; h->Ny = Ny; h->Nz = Nz;
    h->periodic_x = bc_x == AEO_PERIODIC;
    h->periodic_y = bc_y == AEO_PERIODIC;
    h->periodic_z = false;
    char err[512] = "";
    h->sp = spectral_create(Nx, Ny, Nz, g_ctx->stream, err, sizeof err);
    if (!h->sp) return fail(AEO_ERR_UNSUPPORTED, "%s", err);
    if (spectral_column_setup(h->sp, dx, dy, lower, upper, hweight, measure, inv_coupling, gauge,
                              bc_x == AEO_NOFLUX, bc_y == AEO_NOFLUX)) {
        spectral_destroy(h->sp);
        return fail(AEO_ERR_HIP, "column solver setup failed");
    }
    int rc = poisson_alloc(h.get());
    if (rc) return rc;
    *out = h.release();
    return AEO_OK;
}

extern "C" int aeo_poisson_source_buffer(aeo_poisson *h, double **dptr) {
    if (!h || !dptr) return fail(AEO_ERR_ARG, "null argument");
    *dptr = h->src;
    return AEO_OK;
}

struct aeo_unet {
    UNet *N = nullptr;
};

static int poisson_run(aeo_poisson *h, double *phi) {
    Timed t("poisson");
    if (h->kind == 4) {
        int it = 0;
        double res = 0, bn = 0;
        int stt = fcg_solve(h->fcg, h->base->mg, h->net ? h->net->N : nullptr, h->mask, h->mode, h->use_guess,
                            g_ctx->stream, phi, h->src, h->tol, h->maxit, &it, &res, &bn);
        if (stt < 0) return fail(AEO_ERR_HIP, "flexible CG: a network pass failed");
        HIPCHK(hipGetLastError());
        h->iters = it;
        h->resid = stt == AEO_ZERO_RHS ? 0.0 : res / bn;
        h->status = stt;
        return AEO_OK;
    }
    if (h->kind == 2) {
        int it = 0;
        double res = 0, bn = 0;
        int stt = mg_pcg_solve(h->mg, g_ctx->stream, phi, h->src, h->tol, h->maxit, &it, &res, &bn);
        HIPCHK(hipGetLastError());
        h->iters = it;
        // solver_stats of MGPreconditionedCG: ‖r‖/‖b‖ (src/Multigrid.jl:965-966)
        h->resid = stt == AEO_ZERO_RHS ? 0.0 : res / bn;
        h->status = stt;
        return AEO_OK;
    }
    if (h->kind == 3) {
        int cyc = 0;
        double rel = 0;
        int stt = mg_cycles_solve(h->mg, g_ctx->stream, phi, h->src, h->tol, h->maxit, &cyc, &rel);
        HIPCHK(hipGetLastError());
        h->iters = cyc;
        h->resid = rel;
        h->status = stt;
        return AEO_OK;
    }
    int rc = h->kind == 0 ? spectral_fft_solve(h->sp, g_ctx->stream, phi, h->src)
                          : spectral_column_solve(h->sp, g_ctx->stream, phi, h->src);
    if (rc) return fail(AEO_ERR_STATE, "solver not set up");
    HIPCHK(hipGetLastError());
    h->iters = 0;
    h->resid = NAN;
    h->status = AEO_DIRECT;
    return AEO_OK;
}

static int mg_common_create(int kind, int nx, int ny, int nz, double dx, double dy, double dz, int bc_x, int bc_y,
                            int bc_z, const double *cx, const double *cy, const double *cz, const double *rhs_scale,
                            int nu1, int nu2, int smoother, double omega, int vprec, double tol, int maxit,
                            aeo_poisson **out) {
    NEED_CTX();
    if (!out) return fail(AEO_ERR_ARG, "null output handle");
    if (nx < 1 || ny < 1 || nz < 1) return fail(AEO_ERR_ARG, "size must be positive");
    for (int bc : {bc_x, bc_y, bc_z})
        if (bc != AEO_PERIODIC && bc != AEO_NOFLUX)
            return fail(AEO_ERR_ARG, "Multigrid: unsupported BC (use periodic or Neumann)");
    if ((cx == nullptr) != (cy == nullptr) || (cx == nullptr) != (cz == nullptr))
        return fail(AEO_ERR_ARG, "coefficients: give all of cx, cy, cz or none");
    if (smoother != 0 && smoother != 1) return fail(AEO_ERR_ARG, "smoother: 0 red-black Gauss-Seidel, 1 Jacobi");
    if (vprec != AEO_F64 && vprec != AEO_F32) return fail(AEO_ERR_ARG, "bad V-cycle precision");
    if (kind == 3 && vprec != AEO_F64) return fail(AEO_ERR_UNSUPPORTED, "plain multigrid cycles run in FP64");
    if (nu1 < 0 || nu2 < 0 || maxit < 0 || !(tol >= 0)) return fail(AEO_ERR_ARG, "bad sweep count, tolerance or cap");
    if ((double)nx * ny * nz * 8.0 >= 2147483648.0) return fail(AEO_ERR_UNSUPPORTED, "grid exceeds 2 GiB per FP64 array");
    auto h = std::make_unique<aeo_poisson>();
    h->kind = kind; h->Nx = nx; h->Ny = ny; h->Nz = nz;
    h->periodic_x = bc_x == AEO_PERIODIC; h->periodic_y = bc_y == AEO_PERIODIC; h->periodic_z = bc_z == AEO_PERIODIC;
    h->tol = tol; h->maxit = maxit;
    char err[512] = "";
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    h->mg = mg_create(nx, ny, nz, dx, dy, dz, bc_x, bc_y, bc_z, cx, cy, cz, rhs_scale, nu1, nu2, smoother, omega,
                      vprec == AEO_F64 ? 0 : 1, 4, err, sizeof err);
    if (!h->mg) return fail(AEO_ERR_HIP, "%s", err);
    int rc = poisson_alloc(h.get());
    if (rc) return rc;
    *out = h.release();
    return AEO_OK;
}

extern "C" int aeo_poisson_mgpcg_create(int nx, int ny, int nz, double dx, double dy, double dz, int bc_x, int bc_y,
                                        int bc_z, const double *cx, const double *cy, const double *cz,
                                        const double *rhs_scale, int nu1, int nu2, int smoother, double omega,
                                        int vcycle_precision, double tol, int maxit, aeo_poisson **out) {
    return mg_common_create(2, nx, ny, nz, dx, dy, dz, bc_x, bc_y, bc_z, cx, cy, cz, rhs_scale, nu1, nu2, smoother,
                            omega, vcycle_precision, tol, maxit, out);
}

extern "C" int aeo_poisson_mg_create(int nx, int ny, int nz, double dx, double dy, double dz, int bc_x, int bc_y,
                                     int bc_z, const double *cx, const double *cy, const double *cz,
                                     const double *rhs_scale, int nu1, int nu2, double tol, int maxcycles,
                                     aeo_poisson **out) {
    return mg_common_create(3, nx, ny, nz, dx, dy, dz, bc_x, bc_y, bc_z, cx, cy, cz, rhs_scale, nu1, nu2, 0, 1.0,
                            AEO_F64, tol, maxcycles, out);
}

extern "C" int aeo_poisson_mg_set_cycle(aeo_poisson *h, int w_cycle, int fmg) {
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (!h->mg) return fail(AEO_ERR_UNSUPPORTED, "cycle options apply to multigrid solvers");
    if ((w_cycle != 0 && w_cycle != 1) || (fmg != 0 && fmg != 1))
        return fail(AEO_ERR_ARG, "Multigrid: cycle must be :V or :W");
    mg_set_cycle(h->mg, w_cycle, fmg);
    return AEO_OK;
}

extern "C" int aeo_poisson_levels(aeo_poisson *h, int *levels) {
    if (!h || !levels) return fail(AEO_ERR_ARG, "null argument");
    *levels = h->mg ? mg_levels(h->mg) : 1;
    return AEO_OK;
}

extern "C" int aeo_poisson_apply(aeo_poisson *h, double *out, const double *x) {
    NEED_CTX();
    if (!h || !out || !x) return fail(AEO_ERR_ARG, "null argument");
    if (!h->mg) return fail(AEO_ERR_UNSUPPORTED, "aeo_poisson_apply: multigrid solvers only");
    mg_apply(h->mg, g_ctx->stream, out, x);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_poisson_solve_source_buffer(aeo_poisson *h, double *phi) {
    NEED_CTX();
    if (!h || !phi) return fail(AEO_ERR_ARG, "null argument");
    return poisson_run(h, phi);
}

template <typename T>
__global__ void copy_in_kernel(double *__restrict__ buf, const T *__restrict__ f, int Nx, int Ny, int Nz, int H) {
    int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= Nx) return;
    buf[(size_t)i + (size_t)Nx * (j + (size_t)Ny * k)] = (double)f[lin(i + H, j + H, k + H, Nx + 2 * H, Ny + 2 * H)];
}
template <typename T>
__global__ void copy_out_kernel(T *__restrict__ f, const double *__restrict__ buf, int Nx, int Ny, int Nz, int H) {
    int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= Nx) return;
    f[lin(i + H, j + H, k + H, Nx + 2 * H, Ny + 2 * H)] = (T)buf[(size_t)i + (size_t)Nx * (j + (size_t)Ny * k)];
}

extern "C" int aeo_poisson_solve(aeo_poisson *h, int precision, void *p, const void *source, int H) {
    NEED_CTX();
    if (!h || !p || !source || H < 0) return fail(AEO_ERR_ARG, "null argument");
    dim3 grid((h->Nx + 255) / 256, h->Ny, h->Nz);
    if (precision == AEO_F64) hipLaunchKernelGGL(copy_in_kernel<double>, grid, dim3(256), 0, g_ctx->stream, h->src, (const double *)source, h->Nx, h->Ny, h->Nz, H);
    else if (precision == AEO_F32) hipLaunchKernelGGL(copy_in_kernel<float>, grid, dim3(256), 0, g_ctx->stream, h->src, (const float *)source, h->Nx, h->Ny, h->Nz, H);
    else return fail(AEO_ERR_ARG, "bad precision %d", precision);
    int rc = poisson_run(h, h->phi);
    if (rc) return rc;
    if (precision == AEO_F64) hipLaunchKernelGGL(copy_out_kernel<double>, grid, dim3(256), 0, g_ctx->stream, (double *)p, h->phi, h->Nx, h->Ny, h->Nz, H);
    else hipLaunchKernelGGL(copy_out_kernel<float>, grid, dim3(256), 0, g_ctx->stream, (float *)p, h->phi, h->Nx, h->Ny, h->Nz, H);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

// solve!(p, source, solver) on host storage arrays (a CPU Field's data): the
// source's interior gathered on the host into one upload to the source
// buffer, the solve, φ downloaded and scattered into p's interior (p's halo
// untouched, as the reference's solvers leave it). Blocks until p is written.
extern "C" int aeo_poisson_solve_host(aeo_poisson *h, double *p, const double *source, int H) {
    NEED_CTX();
    if (!h || !p || !source || H < 0) return fail(AEO_ERR_ARG, "null argument");
    const size_t Nx = h->Nx, Ny = h->Ny, Nz = h->Nz, sx = Nx + 2 * H, sy = Ny + 2 * H;
    const size_t n = Nx * Ny * Nz;
    std::vector<double> buf(n);
    for (size_t k = 0; k < Nz; k++)
        for (size_t j = 0; j < Ny; j++)
            std::memcpy(&buf[Nx * (j + Ny * k)], &source[H + sx * ((j + H) + sy * (k + H))], sizeof(double) * Nx);
    HIPCHK(hipMemcpyAsync(h->src, buf.data(), sizeof(double) * n, hipMemcpyHostToDevice, g_ctx->stream));
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    int rc = poisson_run(h, h->phi);
    if (rc) return rc;
    HIPCHK(hipMemcpyAsync(buf.data(), h->phi, sizeof(double) * n, hipMemcpyDeviceToHost, g_ctx->stream));
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    for (size_t k = 0; k < Nz; k++)
        for (size_t j = 0; j < Ny; j++)
            std::memcpy(&p[H + sx * ((j + H) + sy * (k + H))], &buf[Nx * (j + Ny * k)], sizeof(double) * Nx);
    return AEO_OK;
}

extern "C" int aeo_poisson_stats(aeo_poisson *h, int *iterations, double *residual, int *status) {
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (iterations) *iterations = h->iters;
    if (residual) *residual = h->resid;
    if (status) *status = h->status;
    return AEO_OK;
}

extern "C" int aeo_poisson_destroy(aeo_poisson *h) {
    if (!h) return AEO_OK;
    if (g_ctx) hipStreamSynchronize(g_ctx->stream);
    spectral_destroy(h->sp);
    mg_destroy(h->mg);
    fcg_destroy(h->fcg);
    hipFree(h->src);
    hipFree(h->phi);
    delete h;
    return AEO_OK;
}

// ---------------------------------------------------------------------------
// cut-cell operators (src/CutCell.jl:602-781), regular grids
// ---------------------------------------------------------------------------
template <typename T>
static int cutcell_call(aeo_grid *g, int op, T *a, T *b, T *c, const T *f0, const T *f1, const T *f2, double *buf,
                        const double *phi, int phi_interior, int bcx, int bcy, int bcz, const double *ax,
                        const double *ay, const double *az, const double *ve, int flag, double s) {
    if (launch_cutcell<T>(g_ctx->stream, op, g->m64, a, b, c, f0, f1, f2, buf, phi, phi_interior, bcx, bcy, bcz, ax,
                          ay, az, ve, flag, s))
        return fail(AEO_ERR_ARG, "bad cut-cell operator");
    HIPCHK(hipGetLastError());
    return AEO_OK;
}
#define CC_CHECK()                                                                                    \
    NEED_CTX();                                                                                       \
    if (!g) return fail(AEO_ERR_ARG, "null grid");                                                    \
    if (g->stretched) return fail(AEO_ERR_UNSUPPORTED, "cut-cell operators: regular grids only");     \
    if (precision != AEO_F64 && precision != AEO_F32) return fail(AEO_ERR_ARG, "bad precision %d", precision)

extern "C" int aeo_cutcell_divergence(aeo_grid *g, int precision, void *div, const void *u, const void *v,
                                      const void *w, const double *ax, const double *ay, const double *az,
                                      const double *vol_eff) {
    CC_CHECK();
    if (!div || !u || !v || !w || !ax || !ay || !az || !vol_eff) return fail(AEO_ERR_ARG, "null argument");
    if (precision == AEO_F64)
        return cutcell_call<double>(g, 0, (double *)div, nullptr, nullptr, (const double *)u, (const double *)v,
                                    (const double *)w, nullptr, nullptr, 0, 0, 0, 0, ax, ay, az, vol_eff, 0, 0);
    return cutcell_call<float>(g, 0, (float *)div, nullptr, nullptr, (const float *)u, (const float *)v,
                               (const float *)w, nullptr, nullptr, 0, 0, 0, 0, ax, ay, az, vol_eff, 0, 0);
}
extern "C" int aeo_cutcell_redistribute(aeo_grid *g, int precision, void *div, const double *vol_eff,
                                        const int *pairs, int npairs) {
    NEED_CTX();
    if (!g || !div || !vol_eff || (npairs > 0 && !pairs)) return fail(AEO_ERR_ARG, "null argument");
    if (npairs < 0) return fail(AEO_ERR_ARG, "npairs must be >= 0");
    if (precision != AEO_F64 && precision != AEO_F32) return fail(AEO_ERR_ARG, "bad precision");
    if (npairs == 0) return AEO_OK;
    const long long nstore = (long long)(g->Nx + 2 * g->H) * (g->Ny + 2 * g->H) * (g->Nz + 2 * g->H);
    if (precision == AEO_F64)
        launch_redistribute<double>(g_ctx->stream, (double *)div, vol_eff, pairs, npairs, nstore);
    else launch_redistribute<float>(g_ctx->stream, (float *)div, vol_eff, pairs, npairs, nstore);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_cutcell_gradient(aeo_grid *g, int precision, void *gx, void *gy, void *gz, const double *p,
                                    const double *ax, const double *ay, const double *az) {
    CC_CHECK();
    if (!gx || !gy || !gz || !p || !ax || !ay || !az) return fail(AEO_ERR_ARG, "null argument");
    if (precision == AEO_F64)
        return cutcell_call<double>(g, 1, (double *)gx, (double *)gy, (double *)gz, nullptr, nullptr, nullptr,
                                    nullptr, p, 0, 0, 0, 0, ax, ay, az, nullptr, 0, 0);
    return cutcell_call<float>(g, 1, (float *)gx, (float *)gy, (float *)gz, nullptr, nullptr, nullptr, nullptr, p, 0,
                               0, 0, 0, ax, ay, az, nullptr, 0, 0);
}
extern "C" int aeo_cutcell_laplacian(aeo_grid *g, int precision, void *out, const void *f, const double *ax,
                                     const double *ay, const double *az, const double *vol_eff, int aperture_power) {
    CC_CHECK();
    if (!out || !f || !ax || !ay || !az || !vol_eff) return fail(AEO_ERR_ARG, "null argument");
    if (aperture_power != 1 && aperture_power != 2) return fail(AEO_ERR_ARG, "aperture_power must be 1 or 2");
    if (precision == AEO_F64)
        return cutcell_call<double>(g, 2, (double *)out, nullptr, nullptr, (const double *)f, nullptr, nullptr,
                                    nullptr, nullptr, 0, 0, 0, 0, ax, ay, az, vol_eff, aperture_power == 2, 0);
    return cutcell_call<float>(g, 2, (float *)out, nullptr, nullptr, (const float *)f, nullptr, nullptr, nullptr,
                               nullptr, 0, 0, 0, 0, ax, ay, az, vol_eff, aperture_power == 2, 0);
}
extern "C" int aeo_cutcell_project_source(aeo_grid *g, int precision, aeo_poisson *solver, const void *u,
                                          const void *v, const void *w, const double *ax, const double *ay,
                                          const double *az, const double *vol_eff) {
    CC_CHECK();
    if (!solver || !u || !v || !w || !ax || !ay || !az || !vol_eff) return fail(AEO_ERR_ARG, "null argument");
    if (solver->Nx != g->Nx || solver->Ny != g->Ny || solver->Nz != g->Nz)
        return fail(AEO_ERR_ARG, "solver and grid sizes differ");
    const int rc = precision == AEO_F64
                       ? cutcell_call<double>(g, 0, nullptr, nullptr, nullptr, (const double *)u, (const double *)v,
                                              (const double *)w, solver->src, nullptr, 0, 0, 0, 0, ax, ay, az,
                                              vol_eff, 1, 0)
                       : cutcell_call<float>(g, 0, nullptr, nullptr, nullptr, (const float *)u, (const float *)v,
                                             (const float *)w, solver->src, nullptr, 0, 0, 0, 0, ax, ay, az,
                                             vol_eff, 1, 0);
    if (rc != AEO_OK) return rc;
    launch_fluid_mean(g_ctx->stream, g->m64, solver->src, vol_eff);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}
extern "C" int aeo_cutcell_project_correct(aeo_grid *g, int precision, void *u, void *v, void *w, const double *phi,
                                           const double *ax, const double *ay, const double *az, int bc_x,
                                           int bc_y, int bc_z, double scale) {
    CC_CHECK();
    if (!u || !v || !w || !phi || !ax || !ay || !az) return fail(AEO_ERR_ARG, "null argument");
    for (int bc : {bc_x, bc_y, bc_z})
        if (bc != AEO_PERIODIC && bc != AEO_NOFLUX) return fail(AEO_ERR_ARG, "φ boundary: periodic or Neumann");
    if (precision == AEO_F64)
        return cutcell_call<double>(g, 1, (double *)u, (double *)v, (double *)w, nullptr, nullptr, nullptr, nullptr,
                                    phi, 1, bc_x, bc_y, bc_z, ax, ay, az, nullptr, 1, scale);
    return cutcell_call<float>(g, 1, (float *)u, (float *)v, (float *)w, nullptr, nullptr, nullptr, nullptr, phi, 1,
                               bc_x, bc_y, bc_z, ax, ay, az, nullptr, 1, scale);
}

// ---------------------------------------------------------------------------
// terrain-following (Gal-Chen) operators and their Poisson solve
// ---------------------------------------------------------------------------
struct aeo_terrain {
    aeo_grid *g;
    TFView v;
    double *d[7] = {};
};

extern "C" int aeo_terrain_create(aeo_grid *g, const double *h_plane, double lid, const double *sigc,
                                  const double *sigf, const double *dzc, const double *dzf, int bc_x, int bc_y,
                                  aeo_terrain **out) {
    NEED_CTX();
    if (!g || !h_plane || !sigc || !sigf || !dzc || !dzf || !out) return fail(AEO_ERR_ARG, "null argument");
    if (g->H < 1) return fail(AEO_ERR_ARG, "the terrain operators need a halo of at least 1");
    for (int bc : {bc_x, bc_y})
        if (bc != AEO_PERIODIC && bc != AEO_NOFLUX) return fail(AEO_ERR_ARG, "lateral maps: periodic or Neumann");
    const int sx = g->Nx + 2 * g->H, sy = g->Ny + 2 * g->H, sz = g->Nz + 2 * g->H;
    double hmax = -1e300;
    for (int q = 0; q < sx * sy; q++) hmax = h_plane[q] > hmax ? h_plane[q] : hmax;
    // terrain_following_grid (src/StretchedGrids.jl:781-783)
    if (!(hmax < lid)) return fail(AEO_ERR_ARG, "terrain height max = %g reaches or exceeds the model lid H = %g", hmax, lid);
    // _slopes (src/StretchedGrids.jl:742-762): centred, one-sided at the outermost ghost ring
    std::vector<double> hx(sx * sy), hy(sx * sy);
    auto H2 = [&](int i, int j) { return h_plane[i + sx * j]; };
    for (int j = 0; j < sy; j++)
        for (int i = 0; i < sx; i++) {
            hx[i + sx * j] = i == 0 ? (H2(1, j) - H2(0, j)) / g->dx
                             : i == sx - 1 ? (H2(sx - 1, j) - H2(sx - 2, j)) / g->dx
                                           : (H2(i + 1, j) - H2(i - 1, j)) / (2 * g->dx);
            hy[i + sx * j] = j == 0 ? (H2(i, 1) - H2(i, 0)) / g->dy
                             : j == sy - 1 ? (H2(i, sy - 1) - H2(i, sy - 2)) / g->dy
                                           : (H2(i, j + 1) - H2(i, j - 1)) / (2 * g->dy);
        }
    auto t = std::make_unique<aeo_terrain>();
    t->g = g;
    const double *src[7] = {h_plane, hx.data(), hy.data(), sigc, sigf, dzc, dzf};
    const size_t len[7] = {(size_t)sx * sy, (size_t)sx * sy, (size_t)sx * sy, (size_t)sz, (size_t)sz, (size_t)sz,
                           (size_t)sz};
    for (int q = 0; q < 7; q++) {
        HIPCHK(hipMalloc(&t->d[q], sizeof(double) * len[q]));
        HIPCHK(upload_dev(t->d[q], src[q], sizeof(double) * len[q]));
    }
    t->v = TFView{t->d[0], t->d[1], t->d[2], t->d[3], t->d[4], t->d[5], t->d[6], lid, g->dx, g->dy,
                  g->Nx, g->Ny, g->Nz, g->H, sx, sy,
                  bc_x == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX, bc_y == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX};
    *out = t.release();
    return AEO_OK;
}
extern "C" int aeo_terrain_destroy(aeo_terrain *t) {
    if (!t) return AEO_OK;
    if (g_ctx) hipStreamSynchronize(g_ctx->stream);
    for (double *p : t->d) hipFree(p);
    delete t;
    return AEO_OK;
}
extern "C" int aeo_terrain_divergence(aeo_terrain *t, double *out, const double *u, const double *v, const double *w) {
    NEED_CTX();
    if (!t || !out || !u || !v || !w) return fail(AEO_ERR_ARG, "null argument");
    launch_tf(g_ctx->stream, 0, t->v, out, u, v, w);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}
extern "C" int aeo_terrain_laplacian(aeo_terrain *t, double *out, const double *f) {
    NEED_CTX();
    if (!t || !out || !f) return fail(AEO_ERR_ARG, "null argument");
    launch_tf(g_ctx->stream, 1, t->v, out, f, nullptr, nullptr);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}
static void terrain_apply_cb(void *ctx, hipStream_t st, double *out, const double *x) {
    launch_tf(st, 2, ((aeo_terrain *)ctx)->v, out, x, nullptr, nullptr);
}
extern "C" int aeo_terrain_apply(aeo_terrain *t, double *out, const double *x) {
    NEED_CTX();
    if (!t || !out || !x) return fail(AEO_ERR_ARG, "null argument");
    terrain_apply_cb(t, g_ctx->stream, out, x);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}
extern "C" int aeo_poisson_terrain_create(aeo_terrain *t, aeo_poisson *base, double tol, int maxit,
                                          aeo_poisson **out) {
    NEED_CTX();
    if (!t || !base || !out) return fail(AEO_ERR_ARG, "null argument");
    if (!base->mg || base->kind != 2) return fail(AEO_ERR_ARG, "the preconditioner must be an MG-preconditioned CG");
    if (base->Nx != t->g->Nx || base->Ny != t->g->Ny || base->Nz != t->g->Nz)
        return fail(AEO_ERR_ARG, "solver and terrain sizes differ");
    if (!(tol >= 0) || maxit < 0) return fail(AEO_ERR_ARG, "bad tolerance or cap");
    auto h = std::make_unique<aeo_poisson>();
    h->kind = 4; h->Nx = base->Nx; h->Ny = base->Ny; h->Nz = base->Nz;
    h->periodic_x = base->periodic_x; h->periodic_y = base->periodic_y; h->periodic_z = false;
    h->base = base; h->mode = 2; h->use_guess = 0; h->tol = tol; h->maxit = maxit;
    FCGOp op;
    op.apply = terrain_apply_cb;
    op.ctx = t;
    h->fcg = fcg_create(base->Nx * base->Ny * base->Nz, op);
    if (!h->fcg) return fail(AEO_ERR_HIP, "allocation failed");
    int rc = poisson_alloc(h.get());
    if (rc) return rc;
    *out = h.release();
    return AEO_OK;
}

// ---------------------------------------------------------------------------
// the anelastic core over Gal-Chen terrain (tfstep.hip)
// ---------------------------------------------------------------------------
struct aeo_tf_stepper {
    aeo_terrain *t;
    aeo_tf_params prm;
    TFWView v;
    size_t n = 0, ni = 0;
    double *us = nullptr, *vs = nullptr, *ws = nullptr, *tn = nullptr;  // predictor and θ' (storage)
    double *snap[4] = {};                                                 // the RK3 step-start state
    double *bx = nullptr, *by = nullptr, *rs = nullptr;                   // the operator's face arrays
    double *work = nullptr;                                               // of the residual checks (interior-sized)
    double *b = nullptr, *phi = nullptr;                                  // source and potential (interior-sized)
    MGPlan *mg = nullptr;
    bool have_phi = false;  // phi holds a previous solve's result (the warm start)
    int iters = 0, status = 0, total_iters = 0;
    double resid = NAN, true_resid = NAN, bnorm = 0, resid0 = NAN;
    // the extrapolated warm start: per substage (0 Euler, 1..3 RK3) the
    // potentials of the last three steps (ph[s][0] the latest), nvalid of them
    double *ph[4][3] = {};
    int nvalid[4] = {};
    double *guess = nullptr;
    // the least-squares guess (warm_start 4): a ring of `basis` earlier
    // (potential, source) pairs, their sources' Gram matrix (host), and the
    // dots' scratch
    double *lx[TFW_KMAX] = {}, *lb[TFW_KMAX] = {};
    int lk = 0, lhead = 0;
    double G[TFW_KMAX][TFW_KMAX] = {};
    double *ppart = nullptr, *pc = nullptr;
    const double *last_b = nullptr;   // the source of the last solve (h->b or a caller's)
    int nsolve = 0;                   // solves since the step began
    int hist_iters[3] = {};           // the iterations and initial residuals of a step's solves
    double hist_r0[3] = {};
};

static void tfw_apply_cb(void *ctx, hipStream_t st, double *out, const double *x) {
    aeo_tf_stepper *h = (aeo_tf_stepper *)ctx;
    Timed tm("tf_apply");
    launch_tfw_apply_march(st, h->v, out, x, nullptr, 0);
}
// L x with the block sums of x·Lx (−1: too many blocks for the slots, no sums)
static int tfw_apply_dot_cb(void *ctx, hipStream_t st, double *out, const double *x, double *part, int cap) {
    aeo_tf_stepper *h = (aeo_tf_stepper *)ctx;
    Timed tm("tf_apply");
    return launch_tfw_apply_march(st, h->v, out, x, part, cap);
}

extern "C" int aeo_tf_stepper_create(aeo_terrain *t, const aeo_tf_params *p, aeo_tf_stepper **out) {
    NEED_CTX();
    if (!t || !p || !out) return fail(AEO_ERR_ARG, "null argument");
    aeo_grid *g = t->g;
    if (g->stretched) return fail(AEO_ERR_UNSUPPORTED, "the terrain core takes a uniform σ spacing");
    if (g->H < 3) return fail(AEO_ERR_ARG, "the terrain core needs a halo of at least 3 (WENO-Z5)");
    if (t->v.bcx != BC_PERIODIC || t->v.bcy != BC_PERIODIC)
        return fail(AEO_ERR_UNSUPPORTED, "the terrain core is periodic in x and y");
    if (p->scheme != AEO_CENTERED && p->scheme != AEO_WENO_Z5)
        return fail(AEO_ERR_UNSUPPORTED, "the terrain core advects with centered or weno_z5");
    if (p->flux_precision != AEO_F64 && p->flux_precision != AEO_F32) return fail(AEO_ERR_ARG, "bad flux precision");
    if (p->vcycle_precision != AEO_F64 && p->vcycle_precision != AEO_F32)
        return fail(AEO_ERR_ARG, "bad V-cycle precision");
    if (p->smoother != 0 && p->smoother != 1) return fail(AEO_ERR_ARG, "smoother: 0 red-black Gauss-Seidel, 1 Jacobi");
    if (!(p->rho0 > 0) || !(p->Hs > 0)) return fail(AEO_ERR_ARG, "the reference density needs rho0 > 0 and Hs > 0");
    if (p->nu1 < 0 || p->nu2 < 0 || p->maxit < 0 || !(p->tol >= 0)) return fail(AEO_ERR_ARG, "bad sweeps, tolerance or cap");
    if (p->warm_start < 0 || p->warm_start > 4) return fail(AEO_ERR_ARG, "warm_start: 0 to 4");
    if (p->warm_start == 4 && (p->basis < 1 || p->basis > TFW_KMAX))
        return fail(AEO_ERR_ARG, "the projection guess keeps 1 to %d solutions", TFW_KMAX);
    auto h = std::make_unique<aeo_tf_stepper>();
    h->t = t;
    h->prm = *p;
    const int Nx = g->Nx, Ny = g->Ny, Nz = g->Nz, H = g->H;
    TFWView &v = h->v;
    v.h = t->d[0]; v.hx = t->d[1]; v.hy = t->d[2];
    v.Hl = t->v.Hl; v.dx = g->dx; v.dy = g->dy; v.dz = g->dz;
    v.rho0 = p->rho0; v.Hs = p->Hs; v.theta0 = p->theta0; v.gamma = p->gamma; v.g_accel = p->g_accel;
    v.Nx = Nx; v.Ny = Ny; v.Nz = Nz; v.H = H; v.sx = Nx + 2 * H; v.sy = Ny + 2 * H; v.buoyancy = p->buoyancy != 0;
    h->n = (size_t)v.sx * v.sy * (Nz + 2 * H);
    h->ni = (size_t)Nx * Ny * Nz;
    const size_t nw = (size_t)Nx * Ny * (Nz + 1);
    for (double **q : {&h->us, &h->vs, &h->ws, &h->tn}) {
        HIPCHK(hipMalloc(q, sizeof(double) * h->n));
        HIPCHK(zero_dev(*q, sizeof(double) * h->n));
    }
    for (double **q : {&h->bx, &h->by, &h->work, &h->b, &h->phi}) {
        HIPCHK(hipMalloc(q, sizeof(double) * h->ni));
        HIPCHK(zero_dev(*q, sizeof(double) * h->ni));
    }
    HIPCHK(hipMalloc(&h->rs, sizeof(double) * nw));
    hipStream_t st = g_ctx->stream;
    launch_tfw_coef(st, v, h->bx, h->by, h->rs);
    // the multigrid on L's 7-point part: face coefficients built on the device, coarsened on the host
    const size_t ncx = (size_t)(Nx + 1) * Ny * Nz, ncy = (size_t)Nx * (Ny + 1) * Nz, ncz = nw;
    double *dcx = nullptr, *dcy = nullptr, *dcz = nullptr;
    HIPCHK(hipMalloc(&dcx, sizeof(double) * ncx));
    HIPCHK(hipMalloc(&dcy, sizeof(double) * ncy));
    HIPCHK(hipMalloc(&dcz, sizeof(double) * ncz));
    launch_tfw_mgcoef(st, v, dcx, dcy, dcz);
    HIPCHK(hipGetLastError());
    std::vector<double> cx(ncx), cy(ncy), cz(ncz);
    HIPCHK(hipMemcpyAsync(cx.data(), dcx, sizeof(double) * ncx, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(cy.data(), dcy, sizeof(double) * ncy, hipMemcpyDeviceToHost, st));
    HIPCHK(hipMemcpyAsync(cz.data(), dcz, sizeof(double) * ncz, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    hipFree(dcx); hipFree(dcy); hipFree(dcz);
    char err[512] = "";
    h->mg = mg_create(Nx, Ny, Nz, g->dx, g->dy, g->dz, AEO_PERIODIC, AEO_PERIODIC, AEO_NOFLUX, cx.data(), cy.data(),
                      cz.data(), nullptr, p->nu1, p->nu2, p->smoother, p->smoother == 1 ? 0.8 : 1.0,
                      p->vcycle_precision == AEO_F64 ? 0 : 1, 4,
                      err, sizeof err);
    if (!h->mg) return fail(AEO_ERR_HIP, "%s", err);
    mg_set_terrain_coef(h->mg, v);
    *out = h.release();
    return AEO_OK;
}

extern "C" int aeo_tf_stepper_destroy(aeo_tf_stepper *h) {
    if (!h) return AEO_OK;
    if (g_ctx) hipStreamSynchronize(g_ctx->stream);
    for (double *q : {h->us, h->vs, h->ws, h->tn, h->bx, h->by, h->rs, h->work, h->b, h->phi})
        if (q) hipFree(q);
    for (double *q : h->snap)
        if (q) hipFree(q);
    for (auto &pair : h->ph)
        for (double *q : pair)
            if (q) hipFree(q);
    if (h->guess) hipFree(h->guess);
    for (double *q : h->lx)
        if (q) hipFree(q);
    for (double *q : h->lb)
        if (q) hipFree(q);
    if (h->ppart) hipFree(h->ppart);
    if (h->pc) hipFree(h->pc);
    if (h->mg) mg_destroy(h->mg);
    delete h;
    return AEO_OK;
}

extern "C" int aeo_tf_fill_halos(aeo_tf_stepper *h, double *u, double *v, double *w, double *theta) {
    NEED_CTX();
    if (!h || !u || !v || !w) return fail(AEO_ERR_ARG, "null argument");
    launch_tfw_halos(g_ctx->stream, h->v, u, v, w, theta);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_tf_tendencies(aeo_tf_stepper *h, double *tu, double *tv, double *tw, double *tt, const double *u,
                                 const double *v, const double *w, const double *theta) {
    NEED_CTX();
    if (!h || !tu || !tv || !tw || !tt || !u || !v || !w || !theta) return fail(AEO_ERR_ARG, "null argument");
    const int sch = h->prm.scheme == AEO_CENTERED ? SCH_CENTERED : SCH_WENO_Z5;
    if (launch_tfw_tendency(g_ctx->stream, h->v, sch, h->prm.flux_precision == AEO_F32, tu, tv, tw, tt,
                            u, v, w, theta, nullptr, 0.0, 0.0, 1.0, 0, 1))
        return fail(AEO_ERR_ARG, "tendency launch failed");
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_tf_divergence(aeo_tf_stepper *h, double *out, const double *u, const double *v, const double *w) {
    NEED_CTX();
    if (!h || !out || !u || !v || !w) return fail(AEO_ERR_ARG, "null argument");
    launch_tfw_div(g_ctx->stream, h->v, h->bx, h->by, h->rs, out, u, v, w);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_tf_gradient(aeo_tf_stepper *h, double *gx, double *gy, double *gw, const double *phi) {
    NEED_CTX();
    if (!h || !gx || !gy || !gw || !phi) return fail(AEO_ERR_ARG, "null argument");
    launch_tfw_grad(g_ctx->stream, h->v, h->bx, h->by, h->rs, gx, gy, gw, phi);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_tf_apply(aeo_tf_stepper *h, double *out, const double *x) {
    NEED_CTX();
    if (!h || !out || !x) return fail(AEO_ERR_ARG, "null argument");
    tfw_apply_cb(h, g_ctx->stream, out, x);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

// the guess from the same substage of the last steps: linear 2a − b, or
// quadratic 3a − 3b + c (c null: linear)
__global__ void tfw_extrapolate_kernel(double *__restrict__ g, const double *__restrict__ a,
                                       const double *__restrict__ b, const double *__restrict__ c, size_t n) {
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x)
        g[t] = c ? 3 * (a[t] - b[t]) + c[t] : 2 * a[t] - b[t];
}

// L φ = b into h->phi (b interior-sized FP64); stage −1: no substage history
static int tfw_solve(aeo_tf_stepper *h, const double *b, int stage = -1) {
    FCGOp op;
    op.apply = tfw_apply_cb;
    op.apply_dot = tfw_apply_dot_cb;
    op.ctx = h;
    hipStream_t st = g_ctx->stream;
    const double *x0 = (h->prm.warm_start && h->have_phi) ? h->phi : nullptr;
    const bool extrap = (h->prm.warm_start == 2 || h->prm.warm_start == 3) && stage >= 0;
    const bool proj = h->prm.warm_start == 4 && stage >= 0;
    const int depth = h->prm.warm_start == 3 ? 3 : 2;
    double gdots[TFW_KMAX + 1] = {};  // b_i·b of the kept pairs, then b·b
    if (proj) {
        x0 = nullptr;
        if (!h->ppart) {
            HIPCHK(hipMalloc(&h->ppart, sizeof(double) * (TFW_KMAX + 1) * 1024));
            HIPCHK(hipMalloc(&h->pc, sizeof(double) * (TFW_KMAX + 1)));
        }
        const int k = h->lk;
        TFBasis X{};
        for (int i = 0; i < k; i++) X.x[i] = h->lb[i];
        X.x[k] = b;
        launch_tfp_dots(st, X, k + 1, b, h->ni, h->ppart, h->pc);
        HIPCHK(hipMemcpyAsync(gdots, h->pc, sizeof(double) * (k + 1), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        if (k > 0 && gdots[k] > 0) {
            // G α = g by Gaussian elimination with partial pivoting on G + δI
            // (δ a 1e-12 fraction of the mean diagonal: near-collinear sources)
            double A[TFW_KMAX][TFW_KMAX + 1];
            double tr = 0;
            for (int i = 0; i < k; i++) tr += h->G[i][i];
            const double delta = 1e-12 * tr / k;
            for (int i = 0; i < k; i++) {
                for (int j = 0; j < k; j++) A[i][j] = h->G[i][j] + (i == j ? delta : 0.0);
                A[i][k] = gdots[i];
            }
            bool ok = true;
            for (int c = 0; c < k && ok; c++) {
                int piv = c;
                for (int r = c + 1; r < k; r++)
                    if (fabs(A[r][c]) > fabs(A[piv][c])) piv = r;
                if (!(fabs(A[piv][c]) > 0)) { ok = false; break; }
                if (piv != c)
                    for (int j = 0; j <= k; j++) std::swap(A[c][j], A[piv][j]);
                for (int r = c + 1; r < k; r++) {
                    const double f = A[r][c] / A[c][c];
                    for (int j = c; j <= k; j++) A[r][j] -= f * A[c][j];
                }
            }
            double alpha[TFW_KMAX] = {};
            for (int r = k - 1; r >= 0 && ok; r--) {
                double v = A[r][k];
                for (int j = r + 1; j < k; j++) v -= A[r][j] * alpha[j];
                alpha[r] = v / A[r][r];
                if (!std::isfinite(alpha[r])) ok = false;
            }
            if (ok) {
                if (!h->guess) HIPCHK(hipMalloc(&h->guess, sizeof(double) * h->ni));
                HIPCHK(hipMemcpy(h->pc, alpha, sizeof(double) * k, hipMemcpyHostToDevice));
                TFBasis Xs{};
                for (int i = 0; i < k; i++) Xs.x[i] = h->lx[i];
                launch_tfp_combine(st, Xs, k, h->pc, h->ni, h->guess);
                x0 = h->guess;
            }
        }
    }
    if (extrap) {
        if (h->nvalid[stage] >= 2) {
            if (!h->guess) HIPCHK(hipMalloc(&h->guess, sizeof(double) * h->ni));
            hipLaunchKernelGGL(tfw_extrapolate_kernel, dim3(2048), dim3(256), 0, st, h->guess,
                               (const double *)h->ph[stage][0], (const double *)h->ph[stage][1],
                               (const double *)(h->nvalid[stage] >= 3 ? h->ph[stage][2] : nullptr), h->ni);
            x0 = h->guess;
        } else if (h->nvalid[stage] == 1) {
            x0 = h->ph[stage][0];
        }
    }
    double bn = 0, res = 0, r0 = 0;
    int it = 0;
    const int stt = mg_pcg_solve_op(h->mg, g_ctx->stream, op, h->phi, b, x0, h->prm.tol, h->prm.maxit, &it, &res, &bn,
                                    nullptr, &r0);
    h->last_b = b;
    h->resid0 = bn > 0 ? r0 / bn : 0.0;
    if (h->nsolve < 3) {
        h->hist_iters[h->nsolve] = it;
        h->hist_r0[h->nsolve] = h->resid0;
    }
    h->nsolve++;
    HIPCHK(hipGetLastError());
    h->have_phi = true;
    if (proj && gdots[h->lk] > 0) {
        // keep (φ, b) in the ring (the oldest pair's slot when full) and
        // the Gram matrix's row and column of the new source
        const int kmax = h->prm.basis, s = h->lk < kmax ? h->lk : h->lhead;
        if (!h->lx[s]) HIPCHK(hipMalloc(&h->lx[s], sizeof(double) * h->ni));
        if (!h->lb[s]) HIPCHK(hipMalloc(&h->lb[s], sizeof(double) * h->ni));
        HIPCHK(hipMemcpyAsync(h->lx[s], h->phi, sizeof(double) * h->ni, hipMemcpyDeviceToDevice, st));
        HIPCHK(hipMemcpyAsync(h->lb[s], b, sizeof(double) * h->ni, hipMemcpyDeviceToDevice, st));
        const int kold = h->lk;
        for (int j = 0; j < kold; j++) {
            if (j == s) continue;
            h->G[s][j] = h->G[j][s] = gdots[j];
        }
        h->G[s][s] = gdots[kold];
        if (h->lk < kmax) h->lk++;
        else h->lhead = (h->lhead + 1) % kmax;
    }
    if (extrap) {
        // the history: each kept potential moves one step older, φ the latest
        double *older = h->ph[stage][depth - 1];
        if (!older) HIPCHK(hipMalloc(&older, sizeof(double) * h->ni));
        for (int q = depth - 1; q > 0; q--) h->ph[stage][q] = h->ph[stage][q - 1];
        h->ph[stage][0] = older;
        HIPCHK(hipMemcpyAsync(older, h->phi, sizeof(double) * h->ni, hipMemcpyDeviceToDevice, st));
        if (h->nvalid[stage] < depth) h->nvalid[stage]++;
    }
    h->iters = it;
    h->total_iters += it;
    h->bnorm = bn;
    h->resid = bn > 0 ? res / bn : 0.0;
    h->true_resid = NAN;  // recomputed on demand (aeo_tf_stats)
    h->status = stt;
    return AEO_OK;
}

extern "C" int aeo_tf_solve(aeo_tf_stepper *h, double *phi, const double *b) {
    NEED_CTX();
    if (!h || !phi || !b) return fail(AEO_ERR_ARG, "null argument");
    HIPCHK(hipMemcpyAsync(h->b, b, sizeof(double) * h->ni, hipMemcpyDeviceToDevice, g_ctx->stream));
    int rc = tfw_solve(h, h->b);
    if (rc) return rc;
    HIPCHK(hipMemcpyAsync(phi, h->phi, sizeof(double) * h->ni, hipMemcpyDeviceToDevice, g_ctx->stream));
    return AEO_OK;
}

// one mass-weighted Euler substage: stage 0 (Euler) or 1..3 of SSP-RK3
static int tfw_substage(aeo_tf_stepper *h, int stage, double *u, double *v, double *w, double *th, double *p,
                        double dt) {
    hipStream_t st = g_ctx->stream;
    double ca = 0, cb = 1;
    int comb = 0;
    stage_coeffs<double>(stage, nullptr, &ca, &cb, &comb);
    {
        Timed tm("tf_halo");
        launch_tfw_halos(st, h->v, u, v, w, th);
    }
    {
        Timed tm("tf_tendency");
        const int sch = h->prm.scheme == AEO_CENTERED ? SCH_CENTERED : SCH_WENO_Z5;
        if (launch_tfw_tendency(st, h->v, sch, h->prm.flux_precision == AEO_F32, h->us, h->vs, h->ws,
                                h->tn, u, v, w, th, h->snap[3], dt, ca, cb, comb, 0))
            return fail(AEO_ERR_ARG, "tendency launch failed");
    }
    {
        Timed tm("tf_halo");
        launch_tfw_halos(st, h->v, h->us, h->vs, h->ws, nullptr);
    }
    {
        Timed tm("tf_div");
        launch_tfw_div(st, h->v, h->bx, h->by, h->rs, h->b, h->us, h->vs, h->ws);
    }
    {
        Timed tm("tf_solve");
        int rc = tfw_solve(h, h->b, stage);
        if (rc) return rc;
    }
    {
        Timed tm("tf_correct");
        launch_tfw_correct(st, h->v, h->bx, h->by, h->rs, u, v, w, th, p, h->us, h->vs, h->ws, h->tn, h->snap[0],
                           h->snap[1], h->snap[2], h->phi, dt, ca, cb, comb);
    }
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_tf_step(aeo_tf_stepper *h, double *u, double *v, double *w, double *theta, double *p, double dt) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta) return fail(AEO_ERR_ARG, "null argument");
    if (!(dt > 0) || !std::isfinite(dt)) return fail(AEO_ERR_ARG, "dt must be positive and finite");
    h->total_iters = 0;
    h->nsolve = 0;
    return tfw_substage(h, 0, u, v, w, theta, p, dt);
}

extern "C" int aeo_tf_step_rk3(aeo_tf_stepper *h, double *u, double *v, double *w, double *theta, double *p,
                               double dt) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta) return fail(AEO_ERR_ARG, "null argument");
    if (!(dt > 0) || !std::isfinite(dt)) return fail(AEO_ERR_ARG, "dt must be positive and finite");
    hipStream_t st = g_ctx->stream;
    for (int q = 0; q < 4; q++)
        if (!h->snap[q]) HIPCHK(hipMalloc(&h->snap[q], sizeof(double) * h->n));
    double *f[4] = {u, v, w, theta};
    for (int q = 0; q < 4; q++)
        HIPCHK(hipMemcpyAsync(h->snap[q], f[q], sizeof(double) * h->n, hipMemcpyDeviceToDevice, st));
    h->total_iters = 0;
    h->nsolve = 0;
    for (int s = 1; s <= 3; s++) {
        int rc = tfw_substage(h, s, u, v, w, theta, s == 3 ? p : nullptr, dt);
        if (rc) return rc;
    }
    return AEO_OK;
}

extern "C" int aeo_tf_project(aeo_tf_stepper *h, double *u, double *v, double *w) {
    NEED_CTX();
    if (!h || !u || !v || !w) return fail(AEO_ERR_ARG, "null argument");
    hipStream_t st = g_ctx->stream;
    launch_tfw_halos(st, h->v, u, v, w, nullptr);
    launch_tfw_div(st, h->v, h->bx, h->by, h->rs, h->b, u, v, w);
    int rc = tfw_solve(h, h->b);
    if (rc) return rc;
    // u = u − Gφ, from copies in the predictor buffers
    HIPCHK(hipMemcpyAsync(h->us, u, sizeof(double) * h->n, hipMemcpyDeviceToDevice, st));
    HIPCHK(hipMemcpyAsync(h->vs, v, sizeof(double) * h->n, hipMemcpyDeviceToDevice, st));
    HIPCHK(hipMemcpyAsync(h->ws, w, sizeof(double) * h->n, hipMemcpyDeviceToDevice, st));
    launch_tfw_correct(st, h->v, h->bx, h->by, h->rs, u, v, w, nullptr, nullptr, h->us, h->vs, h->ws, nullptr,
                       nullptr, nullptr, nullptr, h->phi, 1.0, 0.0, 1.0, 0);
    launch_tfw_halos(st, h->v, u, v, w, nullptr);
    h->have_phi = false;  // φ of a projection is no guess for a step's
    for (int q = 0; q < 4; q++) h->nvalid[q] = 0;
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

// block sums of (b − mb)² and ((b − mb) − ax)² into part[blk], part[nb + blk]
__global__ void tfw_resid_kernel(double *__restrict__ part, const double *__restrict__ b, const double *__restrict__ ax,
                                 double mb, size_t n) {
    __shared__ double sh[2][256];
    double sb = 0.0, se = 0.0;
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
        const double bq = b[t] - mb, e = bq - ax[t];
        sb += bq * bq;
        se += e * e;
    }
    sh[0][threadIdx.x] = sb;
    sh[1][threadIdx.x] = se;
    __syncthreads();
    for (int q = 128; q > 0; q >>= 1) {
        if (threadIdx.x < q) {
            sh[0][threadIdx.x] += sh[0][threadIdx.x + q];
            sh[1][threadIdx.x] += sh[1][threadIdx.x + q];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[blockIdx.x] = sh[0][0];
        part[gridDim.x + blockIdx.x] = sh[1][0];
    }
}
__global__ void tfw_sum_kernel(double *__restrict__ part, const double *__restrict__ b, size_t n) {
    __shared__ double sh[256];
    double s = 0.0;
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) s += b[t];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int q = 128; q > 0; q >>= 1) {
        if (threadIdx.x < q) sh[threadIdx.x] += sh[threadIdx.x + q];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// ‖(b − mean b) − Lφ‖ / ‖b − mean b‖ of the last solve, recomputed in FP64
// from its source (h->b) and solution (h->phi)
static int tfw_true_residual(aeo_tf_stepper *h, double *out) {
    if (!h->last_b) { *out = NAN; return AEO_OK; }
    hipStream_t st = g_ctx->stream;
    constexpr int NB = 512;
    double *d = red_scratch(2 * NB);
    if (!d) return fail(AEO_ERR_HIP, "reduction scratch: out of device memory");
    std::vector<double> hp(2 * NB);
    hipLaunchKernelGGL(tfw_sum_kernel, dim3(NB), dim3(256), 0, st, d, h->last_b, h->ni);
    HIPCHK(hipMemcpyAsync(hp.data(), d, sizeof(double) * NB, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    double mb = 0;
    for (int q = 0; q < NB; q++) mb += hp[q];
    mb /= (double)h->ni;
    tfw_apply_cb(h, st, h->work, h->phi);
    hipLaunchKernelGGL(tfw_resid_kernel, dim3(NB), dim3(256), 0, st, d, h->last_b, (const double *)h->work, mb, h->ni);
    HIPCHK(hipMemcpyAsync(hp.data(), d, sizeof(double) * 2 * NB, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    double bb = 0, rr = 0;
    for (int q = 0; q < NB; q++) {
        bb += hp[q];
        rr += hp[NB + q];
    }
    *out = bb > 0 ? std::sqrt(rr / bb) : 0.0;
    return AEO_OK;
}

extern "C" int aeo_tf_stats(aeo_tf_stepper *h, int *iterations, double *residual, double *true_residual, int *status,
                            int *total_iterations, double *initial_residual) {
    NEED_CTX();
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (initial_residual) *initial_residual = h->resid0;
    if (true_residual) {
        int rc = tfw_true_residual(h, &h->true_resid);
        if (rc) return rc;
    }
    if (iterations) *iterations = h->iters;
    if (residual) *residual = h->resid;
    if (true_residual) *true_residual = h->true_resid;
    if (status) *status = h->status;
    if (total_iterations) *total_iterations = h->total_iters;
    return AEO_OK;
}

extern "C" int aeo_tf_step_history(aeo_tf_stepper *h, int *iterations, double *initial_residuals) {
    if (!h || !iterations || !initial_residuals) return fail(AEO_ERR_ARG, "null argument");
    for (int q = 0; q < 3; q++) {
        iterations[q] = h->hist_iters[q];
        initial_residuals[q] = h->hist_r0[q];
    }
    return AEO_OK;
}

extern "C" int aeo_tf_constraint_residual(aeo_tf_stepper *h, double *u, double *v, double *w, double *out) {
    NEED_CTX();
    if (!h || !u || !v || !w || !out) return fail(AEO_ERR_ARG, "null argument");
    hipStream_t st = g_ctx->stream;
    launch_tfw_halos(st, h->v, u, v, w, nullptr);
    constexpr int NB = 512;
    double *d = red_scratch(NB);
    if (!d) return fail(AEO_ERR_HIP, "reduction scratch: out of device memory");
    launch_tfw_div(st, h->v, h->bx, h->by, h->rs, h->work, u, v, w);
    launch_tfw_absdiv(st, h->v, d, NB, h->work);
    double hb[NB];
    HIPCHK(hipMemcpyAsync(hb, d, sizeof hb, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    double r = 0.0;
    for (int q = 0; q < NB; q++)
        if (hb[q] > r || hb[q] != hb[q]) r = hb[q];
    *out = r;
    return AEO_OK;
}

// ---------------------------------------------------------------------------
// the learned preconditioner
// ---------------------------------------------------------------------------
extern "C" int aeo_unet_create(int nx, int ny, int nz, int in_channels, unsigned long long seed, aeo_unet **out) {
    NEED_CTX();
    if (!out) return fail(AEO_ERR_ARG, "null output handle");
    char err[512] = "";
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    UNet *N = unet_create(nx, ny, nz, in_channels, seed, err, sizeof err);
    if (!N) return fail(AEO_ERR_ARG, "%s", err);
    auto h = new aeo_unet();
    h->N = N;
    *out = h;
    return AEO_OK;
}
extern "C" int aeo_unet_destroy(aeo_unet *h) {
    if (!h) return AEO_OK;
    if (g_ctx) hipStreamSynchronize(g_ctx->stream);
    unet_destroy(h->N);
    delete h;
    return AEO_OK;
}
extern "C" int aeo_unet_num_params(aeo_unet *h, long long *n) {
    if (!h || !n) return fail(AEO_ERR_ARG, "null argument");
    *n = (long long)unet_num_params(h->N);
    return AEO_OK;
}
extern "C" int aeo_unet_get_params(aeo_unet *h, float *host) {
    NEED_CTX();
    if (!h || !host) return fail(AEO_ERR_ARG, "null argument");
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    if (unet_get_params(h->N, host)) return fail(AEO_ERR_HIP, "copy of the parameters failed");
    return AEO_OK;
}
extern "C" int aeo_unet_set_params(aeo_unet *h, const float *host) {
    NEED_CTX();
    if (!h || !host) return fail(AEO_ERR_ARG, "null argument");
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    if (unet_set_params(h->N, g_ctx->stream, host)) return fail(AEO_ERR_HIP, "copy of the parameters failed");
    return AEO_OK;
}
extern "C" int aeo_unet_forward(aeo_unet *h, const double *src, const double *mask, double *out) {
    NEED_CTX();
    if (!h || !src || !out) return fail(AEO_ERR_ARG, "null argument");
    Timed t("unet");
    if (unet_forward(h->N, g_ctx->stream, src, mask, out)) return fail(AEO_ERR_HIP, "U-Net forward failed");
    HIPCHK(hipGetLastError());
    return AEO_OK;
}
extern "C" int aeo_unet_gradients(aeo_unet *h, const double *src, const double *mask, const double *target,
                                  float *grad_host, float *loss) {
    NEED_CTX();
    if (!h || !src || !target || !loss) return fail(AEO_ERR_ARG, "null argument");
    if (unet_gradients(h->N, g_ctx->stream, src, mask, target, grad_host, loss))
        return fail(AEO_ERR_HIP, "U-Net backward failed");
    return AEO_OK;
}
extern "C" int aeo_unet_train_step(aeo_unet *h, const double *src, const double *mask, const double *target, float lr,
                                   float *loss) {
    NEED_CTX();
    if (!h || !src || !target) return fail(AEO_ERR_ARG, "null argument");
    Timed t("unet_train");
    if (unet_train_step(h->N, g_ctx->stream, src, mask, target, lr, loss)) return fail(AEO_ERR_HIP, "training step failed");
    return AEO_OK;
}
extern "C" int aeo_conv3_weight_gradient(int cin, int cout, int nx, int ny, int nz, const void *in, const void *dy,
                                         float *dw, float *db, int *plan) {
    NEED_CTX();
    if (!in || !dy || !dw || !db) return fail(AEO_ERR_ARG, "null argument");
    if (nx < 1 || ny < 1 || nz < 1 || cin < 1 || cout < 1 ||
        (double)nx * ny * nz * (cin > cout ? cin : cout) >= 2147483648.0)
        return fail(AEO_ERR_ARG, "bad extents %d x %d x %d", nx, ny, nz);
    const int rc = conv3_wgrad(g_ctx->stream, cin, cout, nx, ny, nz, in, dy, dw, db, plan);
    if (rc == -1) return fail(AEO_ERR_ARG, "no layer of %d input and %d output channels", cin, cout);
    if (rc) return fail(AEO_ERR_HIP, "weight gradient failed");
    return AEO_OK;
}
extern "C" int aeo_poisson_fcg_create(aeo_poisson *base, aeo_unet *net, const double *mask, int mode, int use_guess,
                                      double tol, int maxit, aeo_poisson **out) {
    NEED_CTX();
    if (!base || !out) return fail(AEO_ERR_ARG, "null argument");
    if (!base->mg || base->kind != 2) return fail(AEO_ERR_ARG, "flexible CG: the base solver must be an MG-preconditioned CG");
    if (mode < 0 || mode > 2) return fail(AEO_ERR_ARG, "mode: 0 network, 1 network + V-cycle, 2 V-cycle");
    if ((mode != 2 || use_guess) && !net) return fail(AEO_ERR_ARG, "flexible CG: this mode needs the network");
    if (!(tol >= 0) || maxit < 0) return fail(AEO_ERR_ARG, "bad tolerance or cap");
    auto h = std::make_unique<aeo_poisson>();
    h->kind = 4; h->Nx = base->Nx; h->Ny = base->Ny; h->Nz = base->Nz;
    h->periodic_x = base->periodic_x; h->periodic_y = base->periodic_y; h->periodic_z = base->periodic_z;
    h->base = base; h->net = net; h->mask = mask; h->mode = mode; h->use_guess = use_guess;
    h->tol = tol; h->maxit = maxit;
    if (net && (unet_dims_match(net->N, base->Nx, base->Ny, base->Nz) == 0))
        return fail(AEO_ERR_ARG, "flexible CG: the network's grid differs from the solver's");
    h->fcg = fcg_create(base->Nx * base->Ny * base->Nz, FCGOp());
    if (!h->fcg) return fail(AEO_ERR_HIP, "flexible CG: allocation failed");
    int rc = poisson_alloc(h.get());
    if (rc) return rc;
    *out = h.release();
    return AEO_OK;
}

// ---------------------------------------------------------------------------
// the stepper
// ---------------------------------------------------------------------------
struct aeo_stepper {
    aeo_grid *g;
    aeo_step_params sp;
    aeo_poisson *solver;
    size_t n;     // storage points
    size_t esz;   // element size
    void *us, *vs, *ws;  // predictor u*
    void *ua, *va, *wa;  // the stage state
    void *ta, *tb;       // θ stage buffers
    double fcor = 0;     // f-plane Coriolis parameter
    void *spg = nullptr; // sponge rate and target vectors (state precision), 5 × (Nz + 2H)
    // static Smagorinsky: νt (storage, state precision), per-level (C_s Δ_k)² and
    // the off-diagonal vertical metric (Nz + 2H each), 1/Pr_t
    void *nut = nullptr, *sgs_lv = nullptr;
    double sgs_s = 0;
};

extern "C" int aeo_stepper_create(aeo_grid *g, const aeo_step_params *sp, aeo_poisson *solver, aeo_stepper **out) {
    NEED_CTX();
    if (!g || !sp || !solver || !out) return fail(AEO_ERR_ARG, "null argument");
    if (sp->precision != AEO_F64 && sp->precision != AEO_F32) return fail(AEO_ERR_ARG, "bad precision");
    int rc = check_scheme(g, sp->mom_scheme, sp->weno_p);
    if (rc) return rc;
    rc = check_scheme(g, sp->scal_scheme, sp->weno_p);
    if (rc) return rc;
    if ((rc = check_step_scheme(sp->mom_scheme)) || (rc = check_step_scheme(sp->scal_scheme))) return rc;
    if (sp->mom_scheme != sp->scal_scheme)
        return fail(AEO_ERR_UNSUPPORTED, "this build advects momentum and θ with one scheme");
    if (solver->Nx != g->Nx || solver->Ny != g->Ny || solver->Nz != g->Nz)
        return fail(AEO_ERR_ARG, "solver size (%d,%d,%d) != grid interior (%d,%d,%d)", solver->Nx, solver->Ny,
                    solver->Nz, g->Nx, g->Ny, g->Nz);
    int bcs[6] = {sp->bc_x, sp->bc_y, sp->bc_z, sp->tbc_x, sp->tbc_y, sp->tbc_z};
    for (int q = 0; q < 6; q++)
        if (!check_bc(bcs[q])) return fail(AEO_ERR_ARG, "bad boundary kind");
    if (sp->bc_x == AEO_WALL || sp->bc_y == AEO_WALL || sp->tbc_x == AEO_WALL || sp->tbc_y == AEO_WALL)
        return fail(AEO_ERR_UNSUPPORTED, "walls are z boundaries");
    // the solver's axes must be the velocity BCs' Poisson kinds (poisson_axis_bcs, :347-354)
    if ((sp->bc_x == AEO_PERIODIC) != solver->periodic_x || (sp->bc_y == AEO_PERIODIC) != solver->periodic_y ||
        (sp->bc_z == AEO_PERIODIC) != solver->periodic_z)
        return fail(AEO_ERR_ARG, "the pressure solver's axis kinds do not match the velocity boundary conditions");
    auto h = std::make_unique<aeo_stepper>();
    h->g = g; h->sp = *sp; h->solver = solver;
    h->n = (size_t)(g->Nx + 2 * g->H) * (g->Ny + 2 * g->H) * (g->Nz + 2 * g->H);
    h->esz = sp->precision == AEO_F64 ? 8 : 4;
    void **bufs[8] = {&h->us, &h->vs, &h->ws, &h->ua, &h->va, &h->wa, &h->ta, &h->tb};
    for (int q = 0; q < 8; q++) {
        HIPCHK(hipMalloc(bufs[q], h->n * h->esz));
        HIPCHK(hipMemsetAsync(*bufs[q], 0, h->n * h->esz, g_ctx->stream));
    }
    *out = h.release();
    return AEO_OK;
}

extern "C" int aeo_stepper_destroy(aeo_stepper *h) {
    if (!h) return AEO_OK;
    if (g_ctx) hipStreamSynchronize(g_ctx->stream);
    void *bufs[8] = {h->us, h->vs, h->ws, h->ua, h->va, h->wa, h->ta, h->tb};
    for (auto b : bufs) hipFree(b);
    if (h->spg) hipFree(h->spg);
    if (h->nut) hipFree(h->nut);
    if (h->sgs_lv) hipFree(h->sgs_lv);
    delete h;
    return AEO_OK;
}

// C_s and Pr_t of BoussinesqSimulation (src/Simulations.jl:237-238, 270):
// the built-in closure StaticSmagorinsky(C_s) of _active_sgs
// (src/operators/sgs_closures.jl:309-318), with sgs_stress = :laplacian
extern "C" int aeo_stepper_set_sgs(aeo_stepper *h, double C_s, double Pr_t) {
    NEED_CTX();
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (!std::isfinite(C_s) || !std::isfinite(Pr_t) || Pr_t == 0)
        return fail(AEO_ERR_ARG, "C_s must be finite and Pr_t finite and non-zero");
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    if (h->sgs_lv) { hipFree(h->sgs_lv); h->sgs_lv = nullptr; }
    if (C_s == 0) return AEO_OK;  // has_sgs = C_s ≠ 0
    const aeo_grid *g = h->g;
    const int n = g->Nz + 2 * g->H;
    std::vector<double> v(2 * (size_t)n, 0.0);
    for (int k = 0; k < n; k++) {
        // _filter_width: (Δx Δy Δz)^(1/3) (UniformZ) or (Δx Δy Δz_c[k])^(1/3) (LevelZ); coef = (C_s Δ)^2
        const double D = g->stretched ? std::pow(g->dx * g->dy * g->dzc[k], 1.0 / 3)
                                      : std::pow(g->dx * g->dy * g->dz, 1.0 / 3);
        const double cd = C_s * D;
        v[k] = cd * cd;
        // _idz_off: 1/Δz (UniformZ) or 2/(Δz_f[k] + Δz_f[k+1]) (LevelZ)
        v[n + k] = g->stretched ? 2 / (g->dzf[k] + g->dzf[k + 1]) : 1 / g->dz;
    }
    if (!h->nut) {
        HIPCHK(hipMalloc(&h->nut, h->n * h->esz));
        HIPCHK(zero_dev(h->nut, h->n * h->esz));
    }
    if (h->sp.precision == AEO_F64) {
        HIPCHK(hipMalloc(&h->sgs_lv, v.size() * sizeof(double)));
        HIPCHK(upload_dev(h->sgs_lv, v.data(), v.size() * sizeof(double)));
    } else {
        std::vector<float> f(v.begin(), v.end());
        HIPCHK(hipMalloc(&h->sgs_lv, f.size() * sizeof(float)));
        HIPCHK(upload_dev(h->sgs_lv, f.data(), f.size() * sizeof(float)));
    }
    h->sgs_s = 1 / Pr_t;
    return AEO_OK;
}

// f_coriolis of BoussinesqSimulation (src/Simulations.jl:269-283): the f-plane
// term of _euler_projection! step 6 (:602-605)
extern "C" int aeo_stepper_set_coriolis(aeo_stepper *h, double f) {
    NEED_CTX();
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (!std::isfinite(f)) return fail(AEO_ERR_ARG, "the Coriolis parameter must be finite");
    h->fcor = f;
    return AEO_OK;
}

// the sponge's per-level vectors in the state precision, 5 × (Nz + 2H): the
// sin² rate of sponge_profile / damping_rate (src/FiniteVolume.jl:524-566)
// at the centre and z-face heights, evaluated once with the reference's
// arithmetic, then the targets of u, v, w (*out = nullptr: sponge off)
static int make_sponge(const aeo_grid *g, int precision, double alpha_max, double z_start, double z_top,
                       const double *zc, const double *zf, const double *target_u, const double *target_v,
                       const double *target_w, void **out) {
    *out = nullptr;
    // has_sponge = α_max ≠ 0 && z_start < z_top; otherwise the sponge is off
    if (alpha_max == 0 || !(z_start < z_top)) return AEO_OK;
    if (!zc || !zf) return fail(AEO_ERR_ARG, "the sponge needs the level heights zc and zf");
    if (!std::isfinite(alpha_max) || !std::isfinite(z_start) || !std::isfinite(z_top))
        return fail(AEO_ERR_ARG, "sponge parameters must be finite");
    const int Nz = g->Nz, H = g->H, sz = Nz + 2 * H;
    const double inv_rise = 1 / (z_top - z_start), half_pi = 0.5 * M_PI;
    auto rate = [&](double xi) {
        if (!(xi >= z_start)) return 0.0;
        const double sn = std::sin(half_pi * (xi - z_start) * inv_rise);
        return alpha_max * sn * sn;
    };
    std::vector<double> v(5 * (size_t)sz, 0.0);
    for (int k = 0; k < Nz; k++) {
        v[H + k] = rate(zc[k]);
        v[sz + H + k] = rate(zf[k]);
        v[2 * sz + H + k] = target_u ? target_u[k] : 0.0;
        v[3 * sz + H + k] = target_v ? target_v[k] : 0.0;
        v[4 * sz + H + k] = target_w ? target_w[k] : 0.0;
    }
    void *d = nullptr;
    if (precision == AEO_F64) {
        HIPCHK(hipMalloc(&d, v.size() * sizeof(double)));
        HIPCHK(upload_dev(d, v.data(), v.size() * sizeof(double)));
    } else {
        std::vector<float> f(v.begin(), v.end());
        HIPCHK(hipMalloc(&d, f.size() * sizeof(float)));
        HIPCHK(upload_dev(d, f.data(), f.size() * sizeof(float)));
    }
    *out = d;
    return AEO_OK;
}

// sponge_α_max, sponge_z_start, sponge_target of BoussinesqSimulation
// (src/Simulations.jl:272-274, 334-352) and add_velocity_sponge! (:375-381)
extern "C" int aeo_stepper_set_sponge(aeo_stepper *h, double alpha_max, double z_start, double z_top,
                                      const double *zc, const double *zf, const double *target_u,
                                      const double *target_v, const double *target_w) {
    NEED_CTX();
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (h->spg) {
        HIPCHK(hipStreamSynchronize(g_ctx->stream));
        hipFree(h->spg);
        h->spg = nullptr;
    }
    return make_sponge(h->g, h->sp.precision, alpha_max, z_start, z_top, zc, zf, target_u, target_v, target_w,
                       &h->spg);
}

template <typename T>
__global__ void copy_interior_kernel(T *__restrict__ dst, const T *__restrict__ src, int Nx, int Ny, int Nz, int H) {
    int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= Nx) return;
    size_t c = lin(i + H, j + H, k + H, Nx + 2 * H, Ny + 2 * H);
    dst[c] = src[c];
}

// One projected forward-Euler substage (_euler_projection!, src/Simulations.jl:
// 531-650) in the buffers of the RK3 driver; stage 0 is step!'s plain Euler.
template <typename T>
static int substage(aeo_stepper *h, int stage, T *u, T *v, T *w, T *th, T *p, double dt) {
    aeo_grid *g = h->g;
    const aeo_step_params &sp = h->sp;
    hipStream_t st = g_ctx->stream;
    const int Nx = g->Nx, Ny = g->Ny, Nz = g->Nz, H = g->H;
    T *us = (T *)h->us, *vs = (T *)h->vs, *ws = (T *)h->ws;
    T *ua = (T *)h->ua, *va = (T *)h->va, *wa = (T *)h->wa;
    T *ta = (T *)h->ta, *tb = (T *)h->tb;
    // inputs and outputs of this substage (the step-start state is the caller's)
    T *ui = stage <= 1 ? u : ua, *vi = stage <= 1 ? v : va, *wi = stage <= 1 ? w : wa;
    T *ti = stage <= 1 ? th : (stage == 2 ? ta : tb);
    T *to = stage == 0 ? ta : (stage == 1 ? ta : (stage == 2 ? tb : th));
    T *uo = (stage == 0 || stage == 3) ? u : ua, *vo = (stage == 0 || stage == 3) ? v : va,
      *wo = (stage == 0 || stage == 3) ? w : wa;
    {
        Timed t("halo");
        HaloSet<T> hs{};
        hs.add(ui, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(vi, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(wi, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(ti, LOC_CC, sp.tbc_x, sp.tbc_y, sp.tbc_z);
        launch_halo_multi<T>(st, hs, Nx, Ny, Nz, H);
    }
    StepPhys ph{sp.nu,       dt, sp.theta0, sp.g_accel, sp.flux_bot, sp.flux_top, g->idzc[H], g->idzc[H + Nz - 1],
                h->fcor, h->spg};
    if (h->sgs_lv) {
        // the closure's νt from the stage state, then its halo (the velocity BCs at a cell centre)
        Timed t("sgs");
        const int n = Nz + 2 * H;
        launch_smag_nut<T>(st, metrics<T>(g), (T *)h->nut, ui, vi, wi, (const T *)h->sgs_lv,
                           (const T *)h->sgs_lv + n);
        int bx = sp.bc_x == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        int by = sp.bc_y == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        int bz = sp.bc_z == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        launch_halo<T>(st, (T *)h->nut, Nx, Ny, Nz, H, LOC_CC, bx, by, bz);
    }
    {
        Timed t("tendency");
        if (launch_tendency_step<T>(st, metrics<T>(g), sp.mom_scheme, sp.weno_p, ui, vi, wi, ti, us, vs, ws, to, th,
                                    ph, stage))
            return fail(AEO_ERR_ARG, "tendency launch failed");
    }
    if (h->sgs_lv) {
        // u* += Δt·∂_j(νt ∂_j u_i); θ' += b·Δt·(1/Pr_t)∂_j(νt ∂_j θ), b the θ combination's weight
        Timed t("sgs");
        double ca_, cb_;
        int comb_;
        stage_coeffs<double>(stage, &ph, &ca_, &cb_, &comb_);
        launch_smag_apply<T>(st, metrics<T>(g), us, vs, ws, to, ui, vi, wi, ti, (const T *)h->nut, dt, cb_,
                             h->sgs_s);
    }
    {
        Timed t("halo");
        HaloSet<T> hs{};
        hs.add(us, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(vs, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(ws, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo_multi<T>(st, hs, Nx, Ny, Nz, H);
    }
    int rc = AEO_OK;
    bool fused = false;
    if (h->solver->kind == 1) {
        // the column solver forms ∇·u* inside its forward row transform (no
        // source buffer round trip; the same values as the divergence kernel).
        // It returns -1, having launched nothing, where x is not periodic.
        Timed t("poisson");
        fused = spectral_column_solve_div<T>(h->solver->sp, st, h->solver->phi, us, vs, ws, g->m64) == 0;
        if (fused) {
            HIPCHK(hipGetLastError());
            h->solver->iters = 0;
            h->solver->resid = NAN;
            h->solver->status = AEO_DIRECT;
        }
    }
    if (!fused) {
        {
            Timed t("divergence");
            launch_div_into<T>(st, h->solver->src, us, vs, ws, g->m64);
        }
        rc = poisson_run(h->solver, h->solver->phi);
        if (rc) return rc;
    }
    double ca, cb;
    int combine;
    stage_coeffs<double>(stage, &ph, &ca, &cb, &combine);
    {
        Timed t("correct");
        // φ's halo: the velocity BCs at a cell centre (a wall mirrors)
        int bx = sp.bc_x == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        int by = sp.bc_y == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        int bz = sp.bc_z == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        launch_correct<T>(st, uo, vo, wo, us, vs, ws, u, v, w, h->solver->phi, p, g->m64, bx, by, bz, ca, cb, combine, dt);
    }
    if (stage == 3) {
        // the halo shell of the combined state (_shell_map!, src/Simulations.jl:741, 693)
        Timed t("shell");
        ShellSet<T> ss{};
        ss.add(u, us, u);
        ss.add(v, vs, v);
        ss.add(w, ws, w);
        ss.add(th, ti, th);
        launch_shell<T>(st, ss, Nx, Ny, Nz, H, ca, cb);
    }
    if (stage == 0) {
        // step!: u's halo holds u*'s fill; θ advanced in place over the interior
        Timed t("shell");
        ShellSet<T> ss{};
        ss.add(u, us, u);
        ss.add(v, vs, v);
        ss.add(w, ws, w);
        launch_shell<T>(st, ss, Nx, Ny, Nz, H, 0.0, 1.0);
        dim3 grid((Nx + 255) / 256, Ny, Nz);
        hipLaunchKernelGGL(copy_interior_kernel<T>, grid, dim3(256), 0, st, th, ta, Nx, Ny, Nz, H);
    }
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

template <typename T>
static int run_step(aeo_stepper *h, void *u, void *v, void *w, void *th, void *p, double dt, bool rk3) {
    if (!rk3) return substage<T>(h, 0, (T *)u, (T *)v, (T *)w, (T *)th, (T *)p, dt);
    // p = φ/Δt of the third stage is the step's pressure; stages 1 and 2 would
    // write values that nothing reads before the third overwrites them
    for (int s = 1; s <= 3; s++) {
        int rc = substage<T>(h, s, (T *)u, (T *)v, (T *)w, (T *)th, s == 3 ? (T *)p : nullptr, dt);
        if (rc) return rc;
    }
    return AEO_OK;
}

extern "C" int aeo_step_rk3(aeo_stepper *h, void *u, void *v, void *w, void *theta, void *p, double dt) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta) return fail(AEO_ERR_ARG, "null argument");
    if (!(dt > 0) || !std::isfinite(dt)) return fail(AEO_ERR_ARG, "dt must be positive and finite");
    return h->sp.precision == AEO_F64 ? run_step<double>(h, u, v, w, theta, p, dt, true)
                                      : run_step<float>(h, u, v, w, theta, p, dt, true);
}

extern "C" int aeo_step_euler(aeo_stepper *h, void *u, void *v, void *w, void *theta, void *p, double dt) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta) return fail(AEO_ERR_ARG, "null argument");
    if (!(dt > 0) || !std::isfinite(dt)) return fail(AEO_ERR_ARG, "dt must be positive and finite");
    return h->sp.precision == AEO_F64 ? run_step<double>(h, u, v, w, theta, p, dt, false)
                                      : run_step<float>(h, u, v, w, theta, p, dt, false);
}

// ---------------------------------------------------------------------------
// the sound-proof (mass-weighted) core, regular grids
// ---------------------------------------------------------------------------
struct aeo_mw_stepper {
    aeo_grid *g;
    aeo_mw_params sp;
    aeo_poisson *solver;
    size_t n, esz;
    void *us, *vs, *ws, *tn;
    void *snap[4] = {};  // the step-start state of step_rk3 (allocated on first use)
    double fcor = 0;     // f-plane Coriolis parameter
    void *spg = nullptr; // sponge vectors, as the Boussinesq stepper's
    // the Smagorinsky closure: νt and κt = νt/Pr_t (storage), per-level (C_s Δ)² and 1/Δz
    void *nut = nullptr, *kap = nullptr, *sgs_lv = nullptr;
    double Pr_t = 0;
    double *Wc = nullptr, *Wf = nullptr, *thf = nullptr;  // device, Nz + 2H
};

extern "C" int aeo_mw_stepper_create(aeo_grid *g, const aeo_mw_params *sp, const double *Wc, const double *Wf,
                                     const double *thetabar_f, aeo_poisson *solver, aeo_mw_stepper **out) {
    NEED_CTX();
    if (!g || !sp || !Wc || !Wf || !thetabar_f || !solver || !out) return fail(AEO_ERR_ARG, "null argument");
    if (g->stretched) return fail(AEO_ERR_UNSUPPORTED, "the sound-proof core runs on regular grids");
    if (g->H < 1) return fail(AEO_ERR_ARG, "the sound-proof core needs a halo of at least 1");
    if (sp->precision != AEO_F64 && sp->precision != AEO_F32) return fail(AEO_ERR_ARG, "bad precision");
    if (solver->Nx != g->Nx || solver->Ny != g->Ny || solver->Nz != g->Nz)
        return fail(AEO_ERR_ARG, "solver and grid sizes differ");
    int bcs[6] = {sp->bc_x, sp->bc_y, sp->bc_z, sp->tbc_x, sp->tbc_y, sp->tbc_z};
    for (int q = 0; q < 6; q++)
        if (!check_bc(bcs[q])) return fail(AEO_ERR_ARG, "bad boundary kind");
    if (sp->bc_x == AEO_WALL || sp->bc_y == AEO_WALL) return fail(AEO_ERR_UNSUPPORTED, "walls are z boundaries");
    if ((sp->bc_x == AEO_PERIODIC) != solver->periodic_x || (sp->bc_y == AEO_PERIODIC) != solver->periodic_y ||
        (sp->bc_z == AEO_PERIODIC) != solver->periodic_z)
        return fail(AEO_ERR_ARG, "the pressure solver's axis kinds do not match the velocity boundary conditions");
    const int nz = g->Nz + 2 * g->H;
    for (int k = 0; k < nz; k++)
        if (!(Wc[k] > 0) || !(Wf[k] > 0) || !(thetabar_f[k] > 0))
            return fail(AEO_ERR_ARG, "reference profiles must be strictly positive");
    auto h = std::make_unique<aeo_mw_stepper>();
    h->g = g; h->sp = *sp; h->solver = solver;
    h->n = (size_t)(g->Nx + 2 * g->H) * (g->Ny + 2 * g->H) * nz;
    h->esz = sp->precision == AEO_F64 ? 8 : 4;
    void **bufs[4] = {&h->us, &h->vs, &h->ws, &h->tn};
    for (int q = 0; q < 4; q++) {
        HIPCHK(hipMalloc(bufs[q], h->n * h->esz));
        HIPCHK(hipMemsetAsync(*bufs[q], 0, h->n * h->esz, g_ctx->stream));
    }
    // the face profile has Nz + 2H + 1 entries addressed (k + 1 at the top level); pad one
    for (double **d : {&h->Wc, &h->Wf, &h->thf}) HIPCHK(hipMalloc(d, sizeof(double) * (nz + 1)));
    std::vector<double> wc(Wc, Wc + nz), wf(Wf, Wf + nz), tf(thetabar_f, thetabar_f + nz);
    wc.push_back(wc.back()); wf.push_back(wf.back()); tf.push_back(tf.back());
    HIPCHK(upload_dev(h->Wc, wc.data(), sizeof(double) * (nz + 1)));
    HIPCHK(upload_dev(h->Wf, wf.data(), sizeof(double) * (nz + 1)));
    HIPCHK(upload_dev(h->thf, tf.data(), sizeof(double) * (nz + 1)));
    *out = h.release();
    return AEO_OK;
}

extern "C" int aeo_mw_stepper_destroy(aeo_mw_stepper *h) {
    if (!h) return AEO_OK;
    if (g_ctx) hipStreamSynchronize(g_ctx->stream);
    for (void *b : {h->us, h->vs, h->ws, h->tn}) hipFree(b);
    for (void *b : h->snap)
        if (b) hipFree(b);
    if (h->spg) hipFree(h->spg);
    for (void *b : {h->nut, h->kap, h->sgs_lv})
        if (b) hipFree(b);
    for (double *b : {h->Wc, h->Wf, h->thf}) hipFree(b);
    delete h;
    return AEO_OK;
}

template <typename T>
static int mw_step(aeo_mw_stepper *h, T *u, T *v, T *w, T *th, T *p, double dt, double ca = 0.0, double cb = 1.0) {
    aeo_grid *g = h->g;
    const aeo_mw_params &sp = h->sp;
    hipStream_t st = g_ctx->stream;
    const int Nx = g->Nx, Ny = g->Ny, Nz = g->Nz, H = g->H;
    T *us = (T *)h->us, *vs = (T *)h->vs, *ws = (T *)h->ws, *tn = (T *)h->tn;
    {
        Timed t("halo");
        HaloSet<T> hs{};
        hs.add(u, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(v, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(w, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(th, LOC_CC, sp.tbc_x, sp.tbc_y, sp.tbc_z);
        launch_halo_multi<T>(st, hs, Nx, Ny, Nz, H);
    }
    MWPhys ph{sp.nu, dt, sp.g_accel, sp.flux_bot * (1 / g->dz), sp.flux_top * (1 / g->dz), sp.buoyancy,
              h->fcor, h->spg};
    if (h->sgs_lv) {
        // νt from the step-start state, its halo with the velocity BCs at a cell centre
        Timed t("sgs");
        const int n = Nz + 2 * H;
        launch_smag_nut<T>(st, metrics<T>(g), (T *)h->nut, u, v, w, (const T *)h->sgs_lv, (const T *)h->sgs_lv + n);
        int bx = sp.bc_x == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        int by = sp.bc_y == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        int bz = sp.bc_z == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        launch_halo<T>(st, (T *)h->nut, Nx, Ny, Nz, H, LOC_CC, bx, by, bz);
    }
    {
        Timed t("tendency");
        launch_mw_tendency<T>(st, metrics<T>(g), us, vs, ws, tn, u, v, w, th, h->Wc, h->Wf, h->thf, ph);
    }
    if (h->sgs_lv) {
        // the W-weighted eddy terms (flux_weights of a sound-proof core), added to the predictor
        Timed t("sgs");
        launch_smag_apply_weighted<T>(st, metrics<T>(g), us, vs, ws, tn, u, v, w, th, (const T *)h->nut, (T *)h->kap,
                                      h->Wc, h->Wf, h->Pr_t, dt);
    }
    {
        Timed t("halo");
        HaloSet<T> hs{};
        hs.add(us, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(vs, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        hs.add(ws, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo_multi<T>(st, hs, Nx, Ny, Nz, H);
    }
    bool fused = false;
    if (h->solver->kind == 1) {
        // the column solver forms the divergence inside its forward row
        // transform (-1, nothing launched, where x is not periodic)
        Timed t("poisson");
        fused = spectral_column_solve_wdiv<T>(h->solver->sp, st, h->solver->phi, us, vs, ws, h->Wc, h->Wf, g->m64) == 0;
        if (fused) {
            HIPCHK(hipGetLastError());
            h->solver->iters = 0;
            h->solver->resid = NAN;
            h->solver->status = AEO_DIRECT;
        }
    }
    if (!fused) {
        {
            Timed t("divergence");
            launch_wdiv<T>(st, g->m64, h->solver->src, (T *)nullptr, us, vs, ws, h->Wc, h->Wf, 0);
        }
        int rc = poisson_run(h->solver, h->solver->phi);
        if (rc) return rc;
    }
    {
        Timed t("correct");
        int bx = sp.bc_x == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        int by = sp.bc_y == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        int bz = sp.bc_z == AEO_PERIODIC ? BC_PERIODIC : BC_NOFLUX;
        // the Runge-Kutta combination c(x, snap) = ca·snap + cb·x of the whole storage in the same passes
        const bool combine = ca != 0.0;
        const T *s0 = combine ? (const T *)h->snap[0] : u, *s1 = combine ? (const T *)h->snap[1] : v;
        const T *s2 = combine ? (const T *)h->snap[2] : w, *s3 = combine ? (const T *)h->snap[3] : th;
        launch_correct<T>(st, u, v, w, us, vs, ws, s0, s1, s2, h->solver->phi, p, g->m64, bx, by, bz, ca, cb, combine,
                          dt, th, tn, s3);
        ShellSet<T> ss{};
        ss.add(u, us, s0);
        ss.add(v, vs, s1);
        ss.add(w, ws, s2);
        if (combine) ss.add(th, th, s3);
        launch_shell<T>(st, ss, Nx, Ny, Nz, H, ca, cb);
    }
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_mw_step(aeo_mw_stepper *h, void *u, void *v, void *w, void *theta, void *p, double dt) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta) return fail(AEO_ERR_ARG, "null argument");
    if (!(dt > 0) || !std::isfinite(dt)) return fail(AEO_ERR_ARG, "dt must be positive and finite");
    return h->sp.precision == AEO_F64
               ? mw_step<double>(h, (double *)u, (double *)v, (double *)w, (double *)theta, (double *)p, dt)
               : mw_step<float>(h, (float *)u, (float *)v, (float *)w, (float *)theta, (float *)p, dt);
}

// f_coriolis and the sponge of a sound-proof core (_build_mass_weighted,
// src/Anelastic.jl:1559-1625; step 6 of _mass_weighted_step!, :1849-1852)
extern "C" int aeo_mw_stepper_set_coriolis(aeo_mw_stepper *h, double f) {
    NEED_CTX();
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (!std::isfinite(f)) return fail(AEO_ERR_ARG, "the Coriolis parameter must be finite");
    h->fcor = f;
    return AEO_OK;
}
extern "C" int aeo_mw_stepper_set_sponge(aeo_mw_stepper *h, double alpha_max, double z_start, double z_top,
                                         const double *zc, const double *zf, const double *target_u,
                                         const double *target_v, const double *target_w) {
    NEED_CTX();
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (h->spg) {
        HIPCHK(hipStreamSynchronize(g_ctx->stream));
        hipFree(h->spg);
        h->spg = nullptr;
    }
    return make_sponge(h->g, h->sp.precision, alpha_max, z_start, z_top, zc, zf, target_u, target_v, target_w,
                       &h->spg);
}

// C_s and Pr_t of a sound-proof core (_build_mass_weighted, src/Anelastic.jl:
// 1559-1625): StaticSmagorinsky(C_s) with the W-weighted SGS fluxes
// (flux_weights, src/operators/sgs_closures.jl:200-217)
extern "C" int aeo_mw_stepper_set_sgs(aeo_mw_stepper *h, double C_s, double Pr_t) {
    NEED_CTX();
    if (!h) return fail(AEO_ERR_ARG, "null argument");
    if (!std::isfinite(C_s) || !std::isfinite(Pr_t) || Pr_t == 0)
        return fail(AEO_ERR_ARG, "C_s must be finite and Pr_t finite and non-zero");
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    if (h->sgs_lv) { hipFree(h->sgs_lv); h->sgs_lv = nullptr; }
    if (C_s == 0) return AEO_OK;
    const aeo_grid *g = h->g;
    const int n = g->Nz + 2 * g->H;
    std::vector<double> v(2 * (size_t)n, 0.0);
    const double D = std::pow(g->dx * g->dy * g->dz, 1.0 / 3);  // _filter_width of UniformZ
    const double cd = C_s * D;
    for (int k = 0; k < n; k++) {
        v[k] = cd * cd;
        v[n + k] = 1 / g->dz;  // _idz_off of UniformZ
    }
    for (void **b : {&h->nut, &h->kap})
        if (!*b) {
            HIPCHK(hipMalloc(b, h->n * h->esz));
            HIPCHK(zero_dev(*b, h->n * h->esz));
        }
    if (h->sp.precision == AEO_F64) {
        HIPCHK(hipMalloc(&h->sgs_lv, v.size() * sizeof(double)));
        HIPCHK(upload_dev(h->sgs_lv, v.data(), v.size() * sizeof(double)));
    } else {
        std::vector<float> f(v.begin(), v.end());
        HIPCHK(hipMalloc(&h->sgs_lv, f.size() * sizeof(float)));
        HIPCHK(upload_dev(h->sgs_lv, f.data(), f.size() * sizeof(float)));
    }
    h->Pr_t = Pr_t;
    return AEO_OK;
}

// step_rk3! of the sound-proof core (src/Anelastic.jl:1905-1945): three
// mass-weighted Euler steps, the second and third combining the whole storage with the start's
template <typename T>
static int mw_rk3(aeo_mw_stepper *h, T *u, T *v, T *w, T *th, T *p, double dt) {
    hipStream_t st = g_ctx->stream;
    for (auto &b : h->snap)
        if (!b) HIPCHK(hipMalloc(&b, h->n * sizeof(T)));
    T *f[4] = {u, v, w, th};
    for (int q = 0; q < 4; q++) HIPCHK(hipMemcpyAsync(h->snap[q], f[q], h->n * sizeof(T), hipMemcpyDeviceToDevice, st));
    int rc;
    const double third = 1.0 / 3;
    if ((rc = mw_step<T>(h, u, v, w, th, p, dt))) return rc;
    if ((rc = mw_step<T>(h, u, v, w, th, p, dt, 0.75, 0.25))) return rc;
    if ((rc = mw_step<T>(h, u, v, w, th, p, dt, third, 2 * third))) return rc;
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

extern "C" int aeo_mw_step_rk3(aeo_mw_stepper *h, void *u, void *v, void *w, void *theta, void *p, double dt) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta) return fail(AEO_ERR_ARG, "null argument");
    if (!(dt > 0) || !std::isfinite(dt)) return fail(AEO_ERR_ARG, "dt must be positive and finite");
    return h->sp.precision == AEO_F64
               ? mw_rk3<double>(h, (double *)u, (double *)v, (double *)w, (double *)theta, (double *)p, dt)
               : mw_rk3<float>(h, (float *)u, (float *)v, (float *)w, (float *)theta, (float *)p, dt);
}

extern "C" int aeo_weighted_divergence(aeo_grid *g, int precision, void *out, const void *u, const void *v,
                                       const void *w, const double *Wc, const double *Wf, int normalize) {
    NEED_CTX();
    if (!g || !out || !u || !v || !w || !Wc || !Wf) return fail(AEO_ERR_ARG, "null argument");
    if (g->stretched) return fail(AEO_ERR_UNSUPPORTED, "weighted_divergence!: regular grids");
    if (precision == AEO_F64)
        launch_wdiv<double>(g_ctx->stream, g->m64, nullptr, (double *)out, (const double *)u, (const double *)v,
                            (const double *)w, Wc, Wf, normalize);
    else if (precision == AEO_F32)
        launch_wdiv<float>(g_ctx->stream, g->m64, nullptr, (float *)out, (const float *)u, (const float *)v,
                           (const float *)w, Wc, Wf, normalize);
    else return fail(AEO_ERR_ARG, "bad precision %d", precision);
    HIPCHK(hipGetLastError());
    return AEO_OK;
}

// ---------------------------------------------------------------------------
// diagnostics and profiling
// ---------------------------------------------------------------------------
static int run_diag(aeo_grid *g, int precision, const void *u, const void *v, const void *w, int what, double *out) {
    NEED_CTX();
    if (!g || !u || !v || !w || !out) return fail(AEO_ERR_ARG, "null argument");
    if (precision != AEO_F64 && precision != AEO_F32) return fail(AEO_ERR_ARG, "bad precision %d", precision);
    constexpr int NB = 512;
    double *d = red_scratch(NB);
    if (!d) return fail(AEO_ERR_HIP, "reduction scratch: out of device memory");
    if (precision == AEO_F64)
        launch_diag<double>(g_ctx->stream, d, NB, (const double *)u, (const double *)v, (const double *)w, g->m64, what);
    else
        launch_diag<float>(g_ctx->stream, d, NB, (const float *)u, (const float *)v, (const float *)w, g->m64, what);
    double h[NB];
    HIPCHK(hipMemcpyAsync(h, d, sizeof h, hipMemcpyDeviceToHost, g_ctx->stream));
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    double r = 0.0;
    for (int b = 0; b < NB; b++) {
        if (what == 2) r += h[b];
        else if (h[b] > r || h[b] != h[b]) r = h[b];
    }
    *out = r;
    return AEO_OK;
}

// The state maxima of cfl_diagnostics (src/TimeIntegration.jl:291-400) on a
// Boussinesq stepper: the velocity halos filled (as the reference does), the
// advective rate max Σ|u_i|/Δx_i; with the Smagorinsky closure, νt from the
// state (compute_sgs!) and its interior maximum (0 without); N from the plane
// means of θ (_brunt_vaisala, :209-232: the largest Boussinesq
// g/θ₀·Δθ̄/Δz_f between consecutive levels, √ of its positive part; 0 without
// buoyancy).
extern "C" int aeo_stepper_cfl(aeo_stepper *h, void *u, void *v, void *w, const void *theta, double *rate,
                               double *nut_max, double *N) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta || !rate || !nut_max || !N) return fail(AEO_ERR_ARG, "null argument");
    aeo_grid *g = h->g;
    const aeo_step_params &sp = h->sp;
    hipStream_t st = g_ctx->stream;
    const int Nx = g->Nx, Ny = g->Ny, Nz = g->Nz, H = g->H;
    const bool f64 = sp.precision == AEO_F64;
    if (f64) {
        launch_halo<double>(st, (double *)u, Nx, Ny, Nz, H, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<double>(st, (double *)v, Nx, Ny, Nz, H, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<double>(st, (double *)w, Nx, Ny, Nz, H, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
    } else {
        launch_halo<float>(st, (float *)u, Nx, Ny, Nz, H, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<float>(st, (float *)v, Nx, Ny, Nz, H, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<float>(st, (float *)w, Nx, Ny, Nz, H, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
    }
    int rc = run_diag(g, sp.precision, u, v, w, 1, rate);
    if (rc) return rc;
    *nut_max = 0;
    if (h->sgs_lv) {
        const int n = Nz + 2 * H;
        if (f64)
            launch_smag_nut<double>(st, g->m64, (double *)h->nut, (const double *)u, (const double *)v,
                                    (const double *)w, (const double *)h->sgs_lv, (const double *)h->sgs_lv + n);
        else
            launch_smag_nut<float>(st, g->m32, (float *)h->nut, (const float *)u, (const float *)v, (const float *)w,
                                   (const float *)h->sgs_lv, (const float *)h->sgs_lv + n);
        rc = run_diag(g, sp.precision, h->nut, h->nut, h->nut, 3, nut_max);
        if (rc) return rc;
    }
    *N = 0;
    if (sp.theta0 != 0) {
        double *d = red_scratch(Nz);
        if (!d) return fail(AEO_ERR_HIP, "reduction scratch: out of device memory");
        if (f64) launch_plane_sum<double>(st, d, (const double *)theta, g->m64);
        else launch_plane_sum<float>(st, d, (const float *)theta, g->m64);
        std::vector<double> sums(Nz);
        HIPCHK(hipMemcpyAsync(sums.data(), d, sizeof(double) * Nz, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        const double np = (double)Nx * Ny;
        double n2max = 0, prev = 0;
        for (int k = 0; k < Nz; k++) {
            const double mean = sums[k] / np;
            if (k > 0) {
                // buoyancy_frequency_squared, Boussinesq form (src/TurbulenceStability.jl:131-132),
                // the plane means Δz_f apart
                const double dzf = g->dzf[H + k];
                const double n2 = (sp.g_accel / sp.theta0) * (mean - prev) * (1 / dzf);
                n2max = (n2 > n2max || n2 != n2) ? n2 : n2max;  // max propagates NaN
            }
            prev = mean;
        }
        *N = n2max != n2max ? n2max : std::sqrt(n2max > 0 ? n2max : 0.0);
    }
    return AEO_OK;
}

// the guard sweep and its reduction over the block partials (NaN-propagating)
static int run_guard(aeo_grid *g, int precision, const void *u, const void *v, const void *w, const void *th,
                     const void *p, const double *Wc, const double *Wf, int *finite, double *div, double *speed) {
    constexpr int NB = 512;
    double *d = red_scratch(3 * NB);
    if (!d) return fail(AEO_ERR_HIP, "reduction scratch: out of device memory");
    if (precision == AEO_F64)
        launch_guard<double>(g_ctx->stream, d, NB, (const double *)u, (const double *)v, (const double *)w,
                             (const double *)th, (const double *)p, Wc, Wf, g->m64);
    else
        launch_guard<float>(g_ctx->stream, d, NB, (const float *)u, (const float *)v, (const float *)w,
                            (const float *)th, (const float *)p, Wc, Wf, g->m64);
    std::vector<double> hp(3 * NB);
    HIPCHK(hipMemcpyAsync(hp.data(), d, sizeof(double) * 3 * NB, hipMemcpyDeviceToHost, g_ctx->stream));
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    double r[3] = {0, 0, 0};
    for (int b = 0; b < NB; b++)
        for (int q = 0; q < 3; q++) {
            const double x = hp[3 * b + q];
            r[q] = (x > r[q] || x != x) ? x : r[q];
        }
    *finite = r[0] == 0;
    *div = r[1];
    *speed = r[2];
    return AEO_OK;
}

// step_guard(sim) (src/TimeIntegration.jl:673-710): the velocity halos filled
// with the stepper's BCs, then finite (every interior u, v, w, θ, p value),
// max |∇·u| and max(|u|, |v|, |w|) in one sweep
extern "C" int aeo_stepper_guard(aeo_stepper *h, void *u, void *v, void *w, const void *theta, const void *p,
                                 int *finite, double *divergence, double *speed) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta || !p || !finite || !divergence || !speed)
        return fail(AEO_ERR_ARG, "null argument");
    aeo_grid *g = h->g;
    const aeo_step_params &sp = h->sp;
    const int Nx = g->Nx, Ny = g->Ny, Nz = g->Nz, H = g->H;
    hipStream_t st = g_ctx->stream;
    if (sp.precision == AEO_F64) {
        launch_halo<double>(st, (double *)u, Nx, Ny, Nz, H, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<double>(st, (double *)v, Nx, Ny, Nz, H, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<double>(st, (double *)w, Nx, Ny, Nz, H, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
    } else {
        launch_halo<float>(st, (float *)u, Nx, Ny, Nz, H, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<float>(st, (float *)v, Nx, Ny, Nz, H, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<float>(st, (float *)w, Nx, Ny, Nz, H, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
    }
    return run_guard(g, sp.precision, u, v, w, theta, p, nullptr, nullptr, finite, divergence, speed);
}

// step_guard(sim::MassWeightedSimulation) (src/Anelastic.jl:2333-2346): the
// divergence is the core's constraint residual max |(1/W_c)∇·(W u)|
// (constraint_residual, :2035-2044), W = ρ̄ (anelastic) or ρ̄θ̄ (pseudo-incompressible)
extern "C" int aeo_mw_stepper_guard(aeo_mw_stepper *h, void *u, void *v, void *w, const void *theta, const void *p,
                                    int *finite, double *divergence, double *speed) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta || !p || !finite || !divergence || !speed)
        return fail(AEO_ERR_ARG, "null argument");
    aeo_grid *g = h->g;
    const aeo_mw_params &sp = h->sp;
    const int Nx = g->Nx, Ny = g->Ny, Nz = g->Nz, H = g->H;
    hipStream_t st = g_ctx->stream;
    if (sp.precision == AEO_F64) {
        launch_halo<double>(st, (double *)u, Nx, Ny, Nz, H, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<double>(st, (double *)v, Nx, Ny, Nz, H, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<double>(st, (double *)w, Nx, Ny, Nz, H, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
    } else {
        launch_halo<float>(st, (float *)u, Nx, Ny, Nz, H, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<float>(st, (float *)v, Nx, Ny, Nz, H, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<float>(st, (float *)w, Nx, Ny, Nz, H, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
    }
    return run_guard(g, sp.precision, u, v, w, theta, p, h->Wc, h->Wf, finite, divergence, speed);
}

// The state maxima of adaptive_dt on a sound-proof core (src/Anelastic.jl:
// 2240-2290): the velocity halos filled, the advective rate; with the
// Smagorinsky closure νt recomputed from the state and its interior maximum
// (0 without); N from the plane means of θ with the local mean θ as the
// reference, (g/θ̄_k)(θ̄_k − θ̄_{k−1})/Δz, θ̄_k = (θ̄_{k−1} + θ̄_k)/2 (0 without buoyancy).
extern "C" int aeo_mw_stepper_cfl(aeo_mw_stepper *h, void *u, void *v, void *w, const void *theta, double *rate,
                                  double *nut_max, double *N) {
    NEED_CTX();
    if (!h || !u || !v || !w || !theta || !rate || !nut_max || !N) return fail(AEO_ERR_ARG, "null argument");
    aeo_grid *g = h->g;
    const aeo_mw_params &sp = h->sp;
    hipStream_t st = g_ctx->stream;
    const int Nx = g->Nx, Ny = g->Ny, Nz = g->Nz, H = g->H;
    const bool f64 = sp.precision == AEO_F64;
    if (f64) {
        launch_halo<double>(st, (double *)u, Nx, Ny, Nz, H, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<double>(st, (double *)v, Nx, Ny, Nz, H, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<double>(st, (double *)w, Nx, Ny, Nz, H, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
    } else {
        launch_halo<float>(st, (float *)u, Nx, Ny, Nz, H, LOC_FX, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<float>(st, (float *)v, Nx, Ny, Nz, H, LOC_FY, sp.bc_x, sp.bc_y, sp.bc_z);
        launch_halo<float>(st, (float *)w, Nx, Ny, Nz, H, LOC_FZ, sp.bc_x, sp.bc_y, sp.bc_z);
    }
    int rc = run_diag(g, sp.precision, u, v, w, 1, rate);
    if (rc) return rc;
    *nut_max = 0;
    if (h->sgs_lv) {
        const int n = Nz + 2 * H;
        if (f64)
            launch_smag_nut<double>(st, g->m64, (double *)h->nut, (const double *)u, (const double *)v,
                                    (const double *)w, (const double *)h->sgs_lv, (const double *)h->sgs_lv + n);
        else
            launch_smag_nut<float>(st, g->m32, (float *)h->nut, (const float *)u, (const float *)v, (const float *)w,
                                   (const float *)h->sgs_lv, (const float *)h->sgs_lv + n);
        rc = run_diag(g, sp.precision, h->nut, h->nut, h->nut, 3, nut_max);
        if (rc) return rc;
    }
    *N = 0;
    if (sp.buoyancy) {
        double *d = red_scratch(Nz);
        if (!d) return fail(AEO_ERR_HIP, "reduction scratch: out of device memory");
        if (f64) launch_plane_sum<double>(st, d, (const double *)theta, g->m64);
        else launch_plane_sum<float>(st, d, (const float *)theta, g->m64);
        std::vector<double> sums(Nz);
        HIPCHK(hipMemcpyAsync(sums.data(), d, sizeof(double) * Nz, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        const double np = (double)Nx * Ny;
        double n2max = 0;
        for (int k = 1; k < Nz; k++) {
            const double lo = sums[k - 1] / np, hi = sums[k] / np;
            const double n2 = (sp.g_accel / ((lo + hi) / 2)) * (hi - lo) * (1 / g->dz);
            n2max = (n2 > n2max || n2 != n2) ? n2 : n2max;
        }
        *N = std::sqrt(n2max);  // NaN stays NaN
    }
    return AEO_OK;
}

extern "C" int aeo_max_divergence(aeo_grid *g, int precision, const void *u, const void *v, const void *w, double *out) {
    return run_diag(g, precision, u, v, w, 0, out);
}
// max_divergence without allocating: the per-level maxima go to the library's
// fixed device array (noalloc.hip) instead of the grown reduction scratch
extern "C" int aeo_max_divergence_noalloc(aeo_grid *g, int precision, const void *u, const void *v, const void *w,
                                          double *out) {
    NEED_CTX();
    if (!g || !u || !v || !w || !out) return fail(AEO_ERR_ARG, "null argument");
    if (precision != AEO_F64 && precision != AEO_F32) return fail(AEO_ERR_ARG, "bad precision %d", precision);
    if (g->Nz > NOALLOC_MAX_LEVELS)
        return fail(AEO_ERR_ARG, "aeo_max_divergence_noalloc serves Nz <= %d (got Nz = %d); use aeo_max_divergence",
                    NOALLOC_MAX_LEVELS, g->Nz);
    double *part = noalloc_scratch(g_ctx->device);
    if (!part) return fail(AEO_ERR_STATE, "no scratch bound on device %d", g_ctx->device);
    if (precision == AEO_F64)
        launch_maxdiv_noalloc<double>(g_ctx->stream, part, (const double *)u, (const double *)v, (const double *)w,
                                      g->m64);
    else
        launch_maxdiv_noalloc<float>(g_ctx->stream, part, (const float *)u, (const float *)v, (const float *)w,
                                     g->m64);
    HIPCHK(hipGetLastError());
    double r = 0.0;
    HIPCHK(hipMemcpyAsync(&r, part + NOALLOC_MAX_LEVELS, sizeof r, hipMemcpyDeviceToHost, g_ctx->stream));
    HIPCHK(hipStreamSynchronize(g_ctx->stream));
    *out = r;
    return AEO_OK;
}
extern "C" int aeo_max_advective_rate(aeo_grid *g, int precision, const void *u, const void *v, const void *w,
                                      double *out) {
    return run_diag(g, precision, u, v, w, 1, out);
}
extern "C" int aeo_kinetic_energy(aeo_grid *g, int precision, const void *u, const void *v, const void *w,
                                  double *out) {
    int rc = run_diag(g, precision, u, v, w, 2, out);
    if (rc == AEO_OK) *out = 0.5 * *out * (g->stretched ? g->dx * g->dy : g->dx * g->dy * g->dz);
    return rc;
}

extern "C" int aeo_launch_levels(const char *kernel, int Nx, int Ny, int Nz, int *levels) {
    if (!kernel || !levels) return fail(AEO_ERR_ARG, "null argument");
    if (Nx < 1 || Ny < 1 || Nz < 1) return fail(AEO_ERR_ARG, "bad extents %d x %d x %d", Nx, Ny, Nz);
    static const struct { const char *name; int (*rule)(int, int, int); } rules[] = {
        {"tendency", chunk_tile}, {"scalar", chunk_brick}, {"limited", chunk_limited},
        {"terrain_tendency", chunk_tfw_tendency}, {"terrain_apply", chunk_tfw_apply},
        {"terrain_smooth", chunk_tf_smooth}, {"terrain_prolong", chunk_tf_prolong}};
    for (const auto &r : rules)
        if (!strcmp(kernel, r.name)) {
            *levels = r.rule(Nx, Ny, Nz);
            return AEO_OK;
        }
    return fail(AEO_ERR_ARG, "no marching kernel named %s", kernel);
}

extern "C" int aeo_profile_enable(int on) {
    NEED_CTX();
    g_ctx->profile = on != 0;
    return AEO_OK;
}
extern "C" int aeo_profile_reset(void) {
    NEED_CTX();
    profile_collect();
    for (auto &kv : g_ctx->prof) {
        kv.second.count = 0;
        kv.second.ms = 0;
    }
    return AEO_OK;
}
extern "C" int aeo_profile_get(const char *kernel, int *count, double *total_ms) {
    NEED_CTX();
    if (!kernel) return fail(AEO_ERR_ARG, "null kernel name");
    profile_collect();
    auto it = g_ctx->prof.find(kernel);
    if (count) *count = it == g_ctx->prof.end() ? 0 : it->second.count;
    if (total_ms) *total_ms = it == g_ctx->prof.end() ? 0 : it->second.ms;
    return AEO_OK;
}
