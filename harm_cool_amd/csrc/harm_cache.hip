// harm_cache.hip -- the cooling-table cache: its file format (cache4d.c:152-326),
// its axis generator (cache4d.c:329-388) and batched lookups on the device,
// one query point per thread (harm_cache.hpp).
//
// File layout (the reference's, byte for byte): the packed 229-byte header,
// the x, y and z axes (double), the values [z][x][y][d] (double) and one
// computed flag per grid point (char; int in "AGACACHE_1.0" files).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/harm_cool.h"
#include "harm_cache.hpp"
#include "harm_host.hpp"

static_assert(sizeof(harm_cache_desc) == 229, "the cache header is the reference's packed 229-byte record");

struct harm_cache {
    harm_cache_desc desc;
    int whole;
    double *vx = nullptr, *vy = nullptr, *vz = nullptr, *values = nullptr;
    uint8_t *counted = nullptr;
    // the splines along y of every component (harm_cache.hpp), or null: formed by the first
    // lookup or solve that reads them (lookup_table)
    mutable std::mutex tab_mu;
    mutable bool tab_tried = false;
    mutable double *tab = nullptr;
    int device = 0;
};

namespace {

constexpr int TPB_C = 256;

#define CCHK(x)                                                                                   \
    do {                                                                                          \
        hipError_t e_ = (x);                                                                      \
        if (e_ != hipSuccess) return harm_host::set_error(std::string(#x) + ": " + hipGetErrorString(e_), 2); \
    } while (0)

size_t npoints(const harm_cache_desc &d) { return (size_t)d.x * d.y * d.z; }

int check_desc(const harm_cache_desc &d)
{
    if (d.x < 1 || d.y < 1 || d.z < 1 || d.d < 1)
        return harm_host::set_error("cache: every axis and the value count must be at least 1", 3);
    if ((double)d.x * d.y * d.z * d.d * 8.0 > 64.0 * (1ull << 30))
        return harm_host::set_error("cache: larger than 64 GiB", 3);
    return 0;
}

bool is_v1(const harm_cache_desc &d) { return std::strncmp(d.ver, "AGACACHE_1.0", 13) == 0; }

// A lookup in z plane zindex >= 0 takes the splines along y from the table; these two
// kernels are the rest: no table, the linear rule, interpolation in z.  plane_too: also
// the points that have a z plane.
__global__ void __launch_bounds__(TPB_C) k_cache_lookup(harm::CacheView c, int mode, uint64_t mask,
                                                        const double *__restrict__ x, const double *__restrict__ y,
                                                        const double *__restrict__ z, const int *__restrict__ zindex,
                                                        double *__restrict__ out, double *__restrict__ dery,
                                                        int *__restrict__ status, size_t n, bool plane_too)
{
    const size_t i = (size_t)blockIdx.x * TPB_C + threadIdx.x;
    if (i >= n) return;
    const int zi = zindex ? zindex[i] : -1;
    if (zi != -1 && !plane_too) return;
    const double zv = z ? z[i] : 0.0;
    const int s = harm::cache_lookup(c, x[i], y[i], zv, zi, mode, mask, out + i, dery ? dery + i : nullptr, n);
    if (status) status[i] = s;
}

__global__ void __launch_bounds__(TPB_C) k_cache_solve_T(harm::CacheView c, const double *__restrict__ rho,
                                                         const double *__restrict__ e,
                                                         const int *__restrict__ zindex, double *__restrict__ T,
                                                         double lo, double hi, int ntrial, double tolf,
                                                         double *__restrict__ berr, int *__restrict__ ret, size_t n,
                                                         bool plane_too)
{
    const size_t i = (size_t)blockIdx.x * TPB_C + threadIdx.x;
    if (i >= n) return;
    const int zi = zindex ? zindex[i] : 0;
    if (zi != -1 && !plane_too) return;
    double t, b;
    const int r = harm::cache_newton_T(e[i], T[i], lo, hi, ntrial, tolf, t, b, [&](double xt, double &v, double &dv) {
        return harm::cache_lookup1<true>(c, rho[i], xt, zi, 0, v, dv) == harm::CACHE_OK;
    });
    T[i] = t;
    if (berr) berr[i] = b;
    if (ret) ret[i] = r;
}

// One (x row, bracket) of component and plane blockIdx.y per thread.
__global__ void __launch_bounds__(TPB_C) k_cache_table(harm::CacheView c, double *__restrict__ tab)
{
    const size_t r = (size_t)blockIdx.x * TPB_C + threadIdx.x;
    const int left = (int)(r / c.X), ix = (int)(r % c.X);
    if (left < 1 || left >= c.Y) return;
    const int zp = (int)blockIdx.y / c.D, k = (int)blockIdx.y % c.D;
    harm::cache_tab_fill(c, zp, k, ix, left, tab + harm::cache_tab_plane(c.X, c.Y) * blockIdx.y);
}

// The axes in LDS (AX: they fit), where a bisection's steps cost a tenth of a global
// read each.
template <bool AX>
__device__ __forceinline__ void stage_axes(const harm::CacheView &c, double *ax, const double *&vx, const double *&vy)
{
    vx = c.vx;
    vy = c.vy;
    if (!AX) return;
    for (int k = threadIdx.x; k < c.X; k += TPB_C) ax[k] = c.vx[k];
    for (int k = threadIdx.x; k < c.Y; k += TPB_C) ax[c.X + k] = c.vy[k];
    __syncthreads();
    vx = ax;
    vy = ax + c.X;
}

// One query per thread, its windows found once and then the components one after
// another.  Bound by the FP64 VALU: 22 divisions and about 300 other operations a
// component with the derivative (2^21 points of a 200x200 table, six values and their
// derivatives: 283 us, 319 a call; with every spline fitted per query, 4300 us a call).
template <bool DER, bool AX>
__global__ void __launch_bounds__(TPB_C) k_lookup_tab(harm::CacheView c, const double *__restrict__ tab, uint64_t mask,
                                                      const double *__restrict__ x, const double *__restrict__ y,
                                                      const double *__restrict__ z, const int *__restrict__ zindex,
                                                      double *__restrict__ out, double *__restrict__ dery,
                                                      int *__restrict__ status, size_t n)
{
    extern __shared__ double ax[];
    const double *vx, *vy;
    stage_axes<AX>(c, ax, vx, vy);
    const size_t i = (size_t)blockIdx.x * TPB_C + threadIdx.x;
    if (i >= n) return;
    const int zi = zindex[i];
    if (zi == -1 && c.Z >= 3) return;  // k_cache_lookup's
    const double xv = x[i], yv = y[i];
    const int lx = harm::cache_bracket(c.X, vx, xv), ly = harm::cache_bracket(c.Y, vy, yv);
    const int s = harm::cache_lookup_status(c, vx, vy, xv, yv, z ? z[i] : 0.0, zi, lx, ly);
    if (status) status[i] = s;
    if (s != harm::CACHE_OK) return;
    const harm::CacheXWin w = harm::cache_xwin(c.X, vx, lx, xv);
    const harm::CacheYWin u = harm::cache_ywin<DER>(c.Y, vy, ly, yv);
    const size_t plane = harm::cache_tab_plane(c.X, c.Y);
    const double *t = tab + plane * c.D * zi;
    for (int k = 0; k < c.D; k++, t += plane) {
        if (!((mask >> k) & 1)) continue;
        double v, dv;
        harm::cache_spline_tab<DER>(c.X, c.Y, t, w, u, v, dv);
        out[k * n + i] = v;
        if (DER) dery[k * n + i] = dv;
    }
}

// One solve per thread, about four trials each (2^21 solves from starts 5% off: 237 us, 256
// a call; with every spline fitted per trial, 1350 us a call).
template <bool AX>
__global__ void __launch_bounds__(TPB_C) k_solve_tab(harm::CacheView c, const double *__restrict__ tab,
                                                     const double *__restrict__ rho, const double *__restrict__ e,
                                                     const int *__restrict__ zindex, double *__restrict__ T, double lo,
                                                     double hi, int ntrial, double tolf, double *__restrict__ berr,
                                                     int *__restrict__ ret, size_t n)
{
    extern __shared__ double ax[];
    const double *vx, *vy;
    stage_axes<AX>(c, ax, vx, vy);
    const size_t i = (size_t)blockIdx.x * TPB_C + threadIdx.x;
    if (i >= n) return;
    const int zi = zindex ? zindex[i] : 0;
    if (zi == -1 && c.Z >= 3) return;  // k_cache_solve_T's
    const double rv = rho[i];
    const int lx = harm::cache_bracket(c.X, vx, rv);
    const harm::CacheXWin w = harm::cache_xwin(c.X, vx, lx, rv);
    const double *t = tab + harm::cache_tab_plane(c.X, c.Y) * c.D * (zi < 0 || zi >= c.Z ? 0 : zi);
    int ly = 0;
    double tn, b;
    const int r = harm::cache_newton_T(e[i], T[i], lo, hi, ntrial, tolf, tn, b, [&](double xt, double &v, double &dv) {
        // the bracket of the trial before, where it still holds this one
        if (ly == 0 || (ly > 1 && xt < vy[ly - 1]) || (ly < c.Y - 1 && !(xt < vy[ly])))
            ly = harm::cache_bracket(c.Y, vy, xt);
        if (harm::cache_lookup_status(c, vx, vy, rv, xt, 0.0, zi, lx, ly) != harm::CACHE_OK) return false;
        harm::cache_spline_tab<true>(c.X, c.Y, t, w, harm::cache_ywin<true>(c.Y, vy, ly, xt), v, dv);
        return true;
    });
    T[i] = tn;
    if (berr) berr[i] = b;
    if (ret) ret[i] = r;
}

harm::CacheView view_of(const harm_cache *c)
{
    return harm::CacheView{c->desc.x, c->desc.y, c->desc.z, c->desc.d, c->desc.xtype, c->desc.ytype, c->desc.ztype,
                           c->whole,  c->vx,     c->vy,     c->vz,     c->values,     c->counted};
}

// Bytes of LDS that both axes take, 0 where they would hold back the occupancy: at
// 16 KiB a block all 8 blocks of 256 threads still fit a CU.
size_t axes_lds(const harm_cache_desc &d)
{
    const size_t b = ((size_t)d.x + d.y) * sizeof(double);
    return b <= 16 * 1024 ? b : 0;
}

// Tables of at most 1 GiB (12 times the values' size) that leave an eighth of the device's
// memory free; larger caches, and those whose table finds no room, are looked up from their
// values.  Formed by the first lookup, not with the cache: the step's caches (one per radius,
// hundreds of them) are never looked up and keep tables of e and p alone with the context.
constexpr size_t TAB_MAX = (size_t)1 << 30;

int form_table(const harm_cache *c, hipStream_t s)
{
    const harm_cache_desc &d = c->desc;
    const size_t planes = (size_t)d.z * d.d, bytes = planes * harm::cache_tab_plane(d.x, d.y) * sizeof(double);
    size_t room = 0, all = 0;
    int dev = -1;
    if (bytes > TAB_MAX || planes > 65535 || hipGetDevice(&dev) != hipSuccess || dev != c->device) return 0;
    if (hipMemGetInfo(&room, &all) != hipSuccess || room < bytes + all / 8) {
        (void)hipGetLastError();
        return 0;
    }
    // another thread's stream capture may not be broken by this thread's allocation
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    CCHK(hipThreadExchangeStreamCaptureMode(&mode));
    double *t = nullptr;
    const hipError_t e = hipMalloc(&t, bytes);
    CCHK(hipThreadExchangeStreamCaptureMode(&mode));
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    const size_t per = (size_t)d.x * d.y;
    hipLaunchKernelGGL(k_cache_table, dim3((unsigned)((per + TPB_C - 1) / TPB_C), (unsigned)planes), dim3(TPB_C), 0, s,
                       view_of(c), t);
    // finished before another thread's stream may read it
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
        (void)hipFree(t);
        return harm_host::set_error("the cache's lookup table could not be formed", 2);
    }
    c->tab = t;
    return 0;
}

// The cache's table, formed on the caller's stream if this is its first use; null: none.
int lookup_table(const harm_cache *c, hipStream_t s, const double *&tab)
{
    std::lock_guard<std::mutex> lk(c->tab_mu);
    int rc = 0;
    if (!c->tab_tried) {
        rc = form_table(c, s);
        c->tab_tried = rc == 0;
    }
    tab = c->tab;
    return rc;
}

}  // namespace

extern "C" {

int harm_cache_axis(int type, int n, double vmin, double vmax, double rat, const double *cust, double *out)
{
    if (n < 1 || !out) return harm_host::set_error("harm_cache_axis: n >= 1 and an output are required", 1);
    double delta;
    switch (type) {
    case HARM_AXIS_LOG:
        delta = (log10(vmax) - log10(vmin)) / (n - 1);
        for (int r = 0; r < n; r++) out[r] = pow(10.0, log10(vmin) + delta * r);
        break;
    case HARM_AXIS_LINEAR:
        delta = (vmax - vmin) / (n - 1);
        for (int r = 0; r < n; r++) out[r] = vmin + delta * r;
        break;
    case HARM_AXIS_NONUNIFORM:
        delta = (vmax - vmin) * (rat - 1.0) / (pow(rat, n) - 1.0) * rat;
        out[0] = vmin;
        for (int r = 1; r < n; r++) {
            out[r] = out[r - 1] + delta;
            delta *= rat;
        }
        break;
    case HARM_AXIS_CUSTOM:
        if (n == 1)
            out[0] = vmin;
        else if (!cust)
            return harm_host::set_error("harm_cache_axis: a custom axis needs its values", 1);
        else
            std::memcpy(out, cust, n * sizeof(double));
        break;
    case HARM_AXIS_ROLLING:
        out[n / 2] = (vmin + vmax) / 2.0;
        for (int r = n / 2 + 1; r < n; r++) out[r] = out[r - 1] * (1.0 + rat);
        for (int r = n / 2 - 1; r >= 0; r--) out[r] = out[r + 1] * (1.0 - rat);
        break;
    default:
        return harm_host::set_error("harm_cache_axis: unknown axis type", 3);
    }
    return 0;
}

int harm_cache_peek(const char *path, harm_cache_desc *desc)
{
    if (!path || !desc) return harm_host::set_error("null argument", 1);
    FILE *f = std::fopen(path, "rb");
    if (!f) return harm_host::set_error(std::string("cannot open ") + path, 4);
    const size_t got = std::fread(desc, sizeof(harm_cache_desc), 1, f);
    std::fclose(f);
    if (got != 1) return harm_host::set_error(std::string("short cache header in ") + path, 4);
    return check_desc(*desc);
}

int harm_cache_read(const char *path, harm_cache_desc *desc, double *vx, double *vy, double *vz, double *values,
                    uint8_t *counted)
{
    if (!vx || !vy || !vz || !values || !counted) return harm_host::set_error("null argument", 1);
    int rc = harm_cache_peek(path, desc);
    if (rc) return rc;
    std::unique_ptr<FILE, int (*)(FILE *)> f(std::fopen(path, "rb"), std::fclose);
    if (!f) return harm_host::set_error(std::string("cannot open ") + path, 4);
    const size_t np = npoints(*desc);
    bool ok = std::fseek(f.get(), sizeof(harm_cache_desc), SEEK_SET) == 0 &&
              std::fread(vx, sizeof(double), desc->x, f.get()) == (size_t)desc->x &&
              std::fread(vy, sizeof(double), desc->y, f.get()) == (size_t)desc->y &&
              std::fread(vz, sizeof(double), desc->z, f.get()) == (size_t)desc->z &&
              std::fread(values, sizeof(double), np * desc->d, f.get()) == np * desc->d;
    if (ok) {
        if (is_v1(*desc)) {  // one int per flag (cache4d.c:209-222)
            std::vector<int> tmp(np);
            ok = std::fread(tmp.data(), sizeof(int), np, f.get()) == np;
            for (size_t i = 0; ok && i < np; i++) counted[i] = (uint8_t)tmp[i];
        } else {
            ok = std::fread(counted, 1, np, f.get()) == np;
        }
    }
    if (!ok) return harm_host::set_error(std::string("short cache file ") + path, 4);
    return 0;
}

int harm_cache_write(const char *path, const harm_cache_desc *desc, const double *vx, const double *vy,
                     const double *vz, const double *values, const uint8_t *counted)
{
    if (!path || !desc || !vx || !vy || !vz || !values || !counted) return harm_host::set_error("null argument", 1);
    int rc = check_desc(*desc);
    if (rc) return rc;
    std::unique_ptr<FILE, int (*)(FILE *)> f(std::fopen(path, "wb"), std::fclose);
    if (!f) return harm_host::set_error(std::string("cannot create ") + path, 4);
    const size_t np = npoints(*desc);
    // the flags are written as chars whatever the header's version (cache4d.c:301-305)
    const bool ok = std::fwrite(desc, sizeof(harm_cache_desc), 1, f.get()) == 1 &&
                    std::fwrite(vx, sizeof(double), desc->x, f.get()) == (size_t)desc->x &&
                    std::fwrite(vy, sizeof(double), desc->y, f.get()) == (size_t)desc->y &&
                    std::fwrite(vz, sizeof(double), desc->z, f.get()) == (size_t)desc->z &&
                    std::fwrite(values, sizeof(double), np * desc->d, f.get()) == np * desc->d &&
                    std::fwrite(counted, 1, np, f.get()) == np;
    if (!ok || std::fflush(f.get()) != 0) return harm_host::set_error(std::string("write failed: ") + path, 4);
    return 0;
}

void harm_cache_free(harm_cache *c)
{
    if (!c) return;
    int prev = 0;
    if (hipGetDevice(&prev) == hipSuccess && hipSetDevice(c->device) == hipSuccess) {
        (void)hipFree(c->vx);
        (void)hipFree(c->vy);
        (void)hipFree(c->vz);
        (void)hipFree(c->values);
        (void)hipFree(c->counted);
        (void)hipFree(c->tab);
        (void)hipSetDevice(prev);
    }
    delete c;
}

static int cache_upload(harm_cache *c, const double *vx, const double *vy, const double *vz, const double *values,
                        const uint8_t *counted)
{
    const harm_cache_desc &d = c->desc;
    const size_t np = npoints(d);
    CCHK(hipGetDevice(&c->device));
    CCHK(hipMalloc(&c->vx, d.x * sizeof(double)));
    CCHK(hipMalloc(&c->vy, d.y * sizeof(double)));
    CCHK(hipMalloc(&c->vz, d.z * sizeof(double)));
    CCHK(hipMalloc(&c->values, np * d.d * sizeof(double)));
    CCHK(hipMalloc(&c->counted, np));
    CCHK(hipMemcpy(c->vx, vx, d.x * sizeof(double), hipMemcpyHostToDevice));
    CCHK(hipMemcpy(c->vy, vy, d.y * sizeof(double), hipMemcpyHostToDevice));
    CCHK(hipMemcpy(c->vz, vz, d.z * sizeof(double), hipMemcpyHostToDevice));
    CCHK(hipMemcpy(c->values, values, np * d.d * sizeof(double), hipMemcpyHostToDevice));
    CCHK(hipMemcpy(c->counted, counted, np, hipMemcpyHostToDevice));
    return 0;
}

harm_cache *harm_cache_create(const harm_cache_desc *desc, const double *vx, const double *vy, const double *vz,
                              const double *values, const uint8_t *counted)
{
    if (!desc || !vx || !vy || !vz || !values || !counted) {
        harm_host::set_error("null argument", 1);
        return nullptr;
    }
    if (check_desc(*desc)) return nullptr;
    const harm_cache_desc &d = *desc;
    if (d.mode != 0) {
        harm_host::set_error("harm_cache_create: only a constant-grid cache (mode 0) is looked up by grid", 3);
        return nullptr;
    }
    if (d.x < 3 || d.y < 3 || d.d > 64 || (d.ztype == HARM_AXIS_ROLLING && d.z < 3)) {
        harm_host::set_error("harm_cache_create: x and y need at least 3 points, a rolling z axis 3, and d <= 64", 3);
        return nullptr;
    }
    // Akima's fit needs increasing abscissae at least 1e-12 apart (akima.c:39-43)
    const double *ax[3] = {vx, vy, vz};
    const int an[3] = {d.x, d.y, d.z};
    for (int a = 0; a < 3; a++)
        for (int i = 1; i < an[a]; i++)
            if (!(ax[a][i] - ax[a][i - 1] >= 1e-12)) {
                harm_host::set_error("harm_cache_create: an axis is not increasing by at least 1e-12", 3);
                return nullptr;
            }
    auto *c = new harm_cache;
    c->desc = d;
    const size_t np = npoints(d);
    size_t ones = 0;
    for (size_t i = 0; i < np; i++) ones += counted[i] == 1;
    // a file that says it is whole is taken at its word, as the reference does
    c->whole = d.wholecachecalculated || ones == np;
    if (cache_upload(c, vx, vy, vz, values, counted)) {
        harm_cache_free(c);
        return nullptr;
    }
    return c;
}

harm_cache *harm_cache_open(const char *path)
{
    harm_cache_desc d;
    if (harm_cache_peek(path, &d)) return nullptr;
    const size_t np = npoints(d);
    std::vector<double> vx(d.x), vy(d.y), vz(d.z), values(np * d.d);
    std::vector<uint8_t> counted(np);
    if (harm_cache_read(path, &d, vx.data(), vy.data(), vz.data(), values.data(), counted.data())) return nullptr;
    return harm_cache_create(&d, vx.data(), vy.data(), vz.data(), values.data(), counted.data());
}

}  // extern "C"

// The device view of a cache and its header, for the step's cache EOS.
int harm_cache_view_of(const harm_cache *c, harm::CacheView &v, harm_cache_desc &d, int &device)
{
    if (!c) return harm_host::set_error("null cache", 1);
    v = view_of(c);
    d = c->desc;
    device = c->device;
    return 0;
}

extern "C" {

int harm_cache_info(const harm_cache *c, harm_cache_desc *desc, int *whole)
{
    if (!c) return harm_host::set_error("null cache", 1);
    if (desc) *desc = c->desc;
    if (whole) *whole = c->whole;
    return 0;
}

int harm_cache_lookup(const harm_cache *c, int mode, const int *dimmask, const double *x, const double *y,
                      const double *z, const int *zindex, double *out, double *dery, int *status, size_t n,
                      void *stream)
{
    if (!c) return harm_host::set_error("null cache", 1);
    if (mode != HARM_INTERP_LIN && mode != HARM_INTERP_SPLINE)
        return harm_host::set_error("harm_cache_lookup: mode is HARM_INTERP_LIN or HARM_INTERP_SPLINE", 3);
    if (!n) return 0;
    if (!x || !y || !out || (!z && !zindex)) return harm_host::set_error("harm_cache_lookup: x, y, out and z or a z index are required", 1);
    uint64_t mask = 0;
    for (int k = 0; k < c->desc.d; k++)
        if (!dimmask || dimmask[k]) mask |= 1ull << k;
    const harm::CacheView v = view_of(c);
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)((n + TPB_C - 1) / TPB_C)), block(TPB_C);
    const double *tab = nullptr;
    if (mode == HARM_INTERP_SPLINE && zindex)
        if (const int rc = lookup_table(c, s, tab)) return rc;
    if (tab) {
        const size_t lds = axes_lds(c->desc);
        auto *k = dery ? (lds ? k_lookup_tab<true, true> : k_lookup_tab<true, false>)
                       : (lds ? k_lookup_tab<false, true> : k_lookup_tab<false, false>);
        hipLaunchKernelGGL(k, grid, block, lds, s, v, tab, mask, x, y, z, zindex, out, dery, status, n);
        CCHK(hipGetLastError());
    }
    if (!tab || c->desc.z >= 3) {
        hipLaunchKernelGGL(k_cache_lookup, grid, block, 0, s, v, mode, mask, x, y, z, zindex, out, dery, status, n,
                           !tab);
    }
    CCHK(hipGetLastError());
    CCHK(hipStreamSynchronize(s));
    return 0;
}

int harm_cache_solve_T(const harm_cache *c, const double *rho, const double *e, const int *zindex, double *T,
                       double Tlo, double Thi, int ntrial, double tolf, double *berr, int *ret, size_t n, void *stream)
{
    if (!c) return harm_host::set_error("null cache", 1);
    if (!n) return 0;
    if (!rho || !e || !T) return harm_host::set_error("harm_cache_solve_T: rho, e and T are required", 1);
    if (ntrial < 1) return harm_host::set_error("harm_cache_solve_T: ntrial >= 1", 3);
    if (Tlo == 0. && Thi == 0.) {
        // the reference's bounds TMin (1 + 1e-6), TMax (1 - 1e-6) (cooleos.c:368-369)
        // from the y axis the cache holds (a rolling axis' header range is not it)
        double ends[2];
        CCHK(hipMemcpy(&ends[0], c->vy, sizeof(double), hipMemcpyDeviceToHost));
        CCHK(hipMemcpy(&ends[1], c->vy + (c->desc.y - 1), sizeof(double), hipMemcpyDeviceToHost));
        Tlo = ends[0] * (1. + 1.e-6);
        Thi = ends[1] * (1. - 1.e-6);
    }
    if (!(Tlo < Thi)) return harm_host::set_error("harm_cache_solve_T: needs Tlo < Thi", 3);
    const harm::CacheView v = view_of(c);
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)((n + TPB_C - 1) / TPB_C)), block(TPB_C);
    const double *tab = nullptr;
    if (const int rc = lookup_table(c, s, tab)) return rc;
    if (tab) {
        const size_t lds = axes_lds(c->desc);
        hipLaunchKernelGGL(lds ? k_solve_tab<true> : k_solve_tab<false>, grid, block, lds, s, v, tab, rho, e, zindex,
                           T, Tlo, Thi, ntrial, tolf, berr, ret, n);
        CCHK(hipGetLastError());
    }
    if (!tab || (zindex && c->desc.z >= 3)) {
        hipLaunchKernelGGL(k_cache_solve_T, grid, block, 0, s, v, rho, e, zindex, T, Tlo, Thi, ntrial, tolf, berr, ret,
                           n, !tab);
    }
    CCHK(hipGetLastError());
    CCHK(hipStreamSynchronize(s));
    return 0;
}

}  // extern "C"
