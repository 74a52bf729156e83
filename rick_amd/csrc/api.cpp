// C ABI of librick_hip.so: device-resident plans and the reference's drop-in
// entry points (wstack, phase_correction) plus rick_fft_planes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "rick_internal.h"
#include "rick_tables.h"

using namespace rick;

namespace {

thread_local int g_status = RICK_OK;
thread_local char g_msg[512] = "";

std::atomic<int> g_kernel{RICK_KAISERBESSEL};  // reference Makefile default (Makefile:66-70)
std::atomic<int> g_phase_on{1};                // PHASE_ON (Makefile:56)

int set_error(int code, const char *fmt, ...)
{
    g_status = code;
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_msg, sizeof g_msg, fmt, ap);
    va_end(ap);
    return code;
}
void clear_error()
{
    g_status = RICK_OK;
    g_msg[0] = '\0';
}

}  // namespace

namespace rick {
int set_status(int code, const char *fmt, ...)
{
    g_status = code;
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_msg, sizeof g_msg, fmt, ap);
    va_end(ap);
    return code;
}
void clear_status() { clear_error(); }
}  // namespace rick

namespace {

#define RICK_HIP(call)                                                                        \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return set_error(e_ == hipErrorOutOfMemory ? RICK_ERR_NOMEM : RICK_ERR_DEVICE,    \
                             "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, \
                             __LINE__);                                                       \
    } while (0)

bool is_pow2(int n) { return n > 0 && (n & (n - 1)) == 0; }

struct TileShape {
    int tu, tv;
};
const TileShape kTiles[] = {{64, 64}, {64, 32}, {32, 32}, {128, 32}, {32, 64}};

// Built-in tile of a plan that names none.  64 x 64 duplicates the fewest
// records; grids of few such tiles take 64 x 32, which spreads a hot tile over
// more workgroups (512^2 x 8 planes, 516 k rows: image 171 -> 165 us, 256^2 x 4
// 81 -> 77 us; 1024^2 x 16 with 4096 tiles: 670 -> 677 us), and rows above 4096
// cells 128 x 32, which keeps them at 64 tiles, the row transform's occupancy
// mask (8192^2 x 64 planes: image 23.1 -> 22.6 ms).  GAUSS_HI_PRECISION of support 9 and
// more, whose records cost most, takes 64 x 32 only for tiles that are few and full:
// gridding with 64 x 32 and 64 x 64 tiles, support 9 FP64, 693 rows on 256 x 128 x 2 60
// and 46 us, 50 k rows on 512^2 x 8 84 and 65, on 256^2 x 4 50 and 55.
TileShape default_tile(const rick_plan_desc &d)
{
    if (d.grid_size_x > 4096) return {128, 32};
    const uint64_t nb = (uint64_t)d.num_w_planes * ((d.grid_size_x + 63) / 64) *
                        ((d.grid_size_y + 63) / 64);
    if (d.kernel == RICK_GAUSS_HI_PRECISION && d.w_support >= 9 &&
        (nb > 256 || d.max_points < 128 * nb))
        return {64, 64};
    // 64 x 32 tiles take one workgroup per task, of which a launch holds fewer
    // than 2^32 threads; the larger tiles' workgroups stay and take many.
    const uint64_t rows = d.rows_per_task > 0 ? d.rows_per_task : 512;
    const bool fits = (2 * nb + 4ull * d.max_points / rows + 1) * 512 < (1ull << 32);
    return nb <= 1024 && fits ? TileShape{64, 32} : TileShape{64, 64};
}

}  // namespace

struct rick_plan_s {
    rick_plan_desc d{};
    GridGeom geom{};
    GridWork work{};
    FftPlan fft{};
    PhaseGeom phase{};
    void *dmem = nullptr;
    size_t dbytes = 0;
    double *table_d = nullptr;
    void *tmp_plane = nullptr;
    bool fft_ok = false;    // power-of-two axes in [16, 8192]: the Stockham engine of fft.hip
    bool gen_ok = false;    // any other axis lengths: the mixed-radix / Bluestein engine
    GenFft gen{};
    bool grid_ok = false;
    Timing timing;
};

namespace {

// Checks a description and derives its gridding geometry and launch shape.
int plan_geometry(const rick_plan_desc &d, GridGeom &g)
{
    if (d.num_w_planes < 1 || d.grid_size_x < 1 || d.grid_size_y < 1)
        return set_error(RICK_ERR_INVALID, "bad grid %d x %d x %d planes", d.grid_size_x,
                         d.grid_size_y, d.num_w_planes);
    if (d.kernel < RICK_GAUSS || d.kernel > RICK_GAUSS_HI_PRECISION)
        return set_error(RICK_ERR_INVALID, "unknown kernel kind %d", d.kernel);
    if (d.w_support < 1 || d.w_support > kMaxSupport || (d.w_support % 2) == 0)
        return set_error(RICK_ERR_INVALID, "w_support must be odd and in [1, %d], got %d",
                         kMaxSupport, d.w_support);
    if (d.precision != RICK_FP64 && d.precision != RICK_FP32)
        return set_error(RICK_ERR_INVALID, "unknown precision %d", d.precision);
    if (!(d.dx > 0.0) || !(d.dw > 0.0))
        return set_error(RICK_ERR_INVALID, "dx and dw must be positive");
    if (d.xaxistot < 0 || d.yaxistot < 0)
        return set_error(RICK_ERR_INVALID, "negative image totals %d x %d", d.xaxistot,
                         d.yaxistot);

    int tu = d.tile_u ? d.tile_u : 64, tv = d.tile_v ? d.tile_v : 64;
    if (!d.tile_u && !d.tile_v) {
        const TileShape t = default_tile(d);
        tu = t.tu;
        tv = t.tv;
    }
    bool tile_ok = false;
    for (const auto &t : kTiles) tile_ok |= (t.tu == tu && t.tv == tv);
    if (!tile_ok) return set_error(RICK_ERR_INVALID, "unsupported tile %d x %d", tu, tv);
    if (tu < d.w_support || tv < d.w_support)
        return set_error(RICK_ERR_INVALID, "tile %d x %d smaller than support %d", tu, tv,
                         d.w_support);
    g.planes = d.num_w_planes;
    g.nx = d.grid_size_x;
    g.ny = d.grid_size_y;
    g.support = d.w_support;
    g.kl = (d.w_support - 1) / 2;
    g.kind = d.kernel;
    g.dx = d.dx;
    g.dw = d.dw;
    g.inv_dx = exact_inverse(d.dx);
    g.inv_dw = exact_inverse(d.dw);
    g.tu = tu;
    g.tv = tv;
    g.tu_shift = __builtin_ctz((unsigned)tu);
    g.tv_shift = __builtin_ctz((unsigned)tv);
    g.tiles_u = (g.nx + tu - 1) / tu;
    g.tiles_v = (g.ny + tv - 1) / tv;
    const uint64_t nb = (uint64_t)g.planes * g.tiles_u * g.tiles_v;
    if (nb >= (1ull << 31)) return set_error(RICK_ERR_INVALID, "too many grid tiles");
    g.nb = (uint32_t)nb;
    g.cshift = counter_shift(g.nb);
    g.ntable = kTableOversample * d.w_support;
    // ~64-128 KB of grid per zero task measured best (LOFAR-like grid).
    g.zrun = d.precision == RICK_FP64 ? 2 : 4;
    // Unrolled footprint loops of the tile kernel: the instantiated lengths.
    {
        const int unrolls[] = {7, 9, 11, 15};
        g.smax = 0;
        for (int u : unrolls)
            if (u >= d.w_support && (d.footprint_unroll == 0 ? g.smax == 0 : u == d.footprint_unroll))
                g.smax = u;
        if (g.smax == 0)
            return set_error(RICK_ERR_INVALID,
                             "footprint_unroll %d: must be 0 or one of 7, 9, 11, 15 and >= "
                             "w_support %d", d.footprint_unroll, d.w_support);
    }
    const bool builtin = d.rows_per_task <= 0;
    g.rmax = builtin ? default_rows_per_task(g, d.max_points) : (uint32_t)d.rows_per_task;
    g.rmin = builtin ? kShortestTask : g.rmax;
    if ((uint64_t)d.max_points * 4ull >= (1ull << 32))
        return set_error(RICK_ERR_INVALID, "max_points %u too large (limit 2^30)", d.max_points);

    if (d.max_points > 0) {
        // Built-in tasks are made longer before a plan is refused for their number.
        while (builtin && g.rmin < 4096 && grid_launch_limit(g, d.max_points)) {
            g.rmin *= 2;
            g.rmax = std::max(g.rmax, g.rmin);
        }
        if (const char *why = grid_launch_limit(g, d.max_points))
            return set_error(RICK_ERR_INVALID, "%d x %d x %d grid, %d x %d tiles, %u points: %s",
                             g.nx, g.ny, g.planes, tu, tv, d.max_points, why);
    }
    return RICK_OK;
}

// Device memory of a plan: [table | twiddles x | twiddles y | l table | m table |
// tmp plane | any-size tables and scratch | gridding workspace].
struct PlanLayout {
    bool fft_ok = false, gen_ok = false, grid_ok = false;
    GenFft gen{};
    size_t table = 0, twx = 0, twy = 0, l = 0, m = 0, tmp = 0, gen_tab = 0, gen_work = 0, work = 0,
           bytes = 0;
};
PlanLayout plan_layout(const rick_plan_desc &d, const GridGeom &g)
{
    PlanLayout L;
    L.grid_ok = d.max_points > 0;
    L.fft_ok = is_pow2(g.nx) && is_pow2(g.ny) && g.nx >= 16 && g.ny >= 16 && g.nx <= 8192 &&
               g.ny <= 8192;
    if (!L.fft_ok) L.gen_ok = gen_fft_prepare(g.nx, g.ny, d.precision, &L.gen);
    const size_t csz = d.precision == RICK_FP64 ? 16 : 8;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) / 256 * 256;
        return at;
    };
    L.table = take(sizeof(double) * kMaxTable);
    L.twx = take(csz * (size_t)g.nx);
    L.twy = take(csz * (size_t)g.ny);
    L.l = take(sizeof(double) * (size_t)g.nx);
    L.m = take(sizeof(double) * (size_t)g.ny);
    L.tmp = take(L.fft_ok && fft_needs_tmp(d.precision, g.ny) ? csz * (size_t)g.nx * g.ny : 0);
    L.gen_tab = take(L.gen_ok ? L.gen.table_bytes : 0);
    L.gen_work = take(L.gen_ok ? L.gen.work_bytes : 0);
    L.work = off;
    if (L.grid_ok) off += grid_work_bytes(g, d.max_points, d.precision);
    L.bytes = off;
    return L;
}

}  // namespace

extern "C" {

int rick_last_status(void) { return g_status; }
const char *rick_last_error(void) { return g_msg; }
const char *rick_version(void) { return "rick-mi355x 0.1 (gfx950)"; }

int rick_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int rick_set_kernel(int kind)
{
    clear_error();
    if (kind < RICK_GAUSS || kind > RICK_GAUSS_HI_PRECISION)
        return set_error(RICK_ERR_INVALID, "unknown kernel kind %d", kind);
    g_kernel = kind;
    return RICK_OK;
}
int rick_get_kernel(void) { return g_kernel; }
int rick_set_phase(int on)
{
    clear_error();
    g_phase_on = on ? 1 : 0;
    return RICK_OK;
}
int rick_get_phase(void) { return g_phase_on; }

int rick_plan_destroy(rick_plan p)
{
    if (!p) return RICK_OK;
    int dev = 0;
    hipGetDevice(&dev);
    hipSetDevice(p->d.device);
    if (p->dmem) hipFree(p->dmem);
    for (auto &v : p->timing.ev)
        for (auto &e : v) {
            hipEventDestroy(e.first);
            hipEventDestroy(e.second);
        }
    hipSetDevice(dev);
    delete p;
    return RICK_OK;
}

int rick_plan_create(rick_plan *out, const rick_plan_desc *desc)
{
    clear_error();
    if (!out || !desc) return set_error(RICK_ERR_INVALID, "null plan or descriptor");
    *out = nullptr;
    const rick_plan_desc &d = *desc;
    auto p = std::make_unique<rick_plan_s>();
    p->d = d;
    GridGeom &g = p->geom;
    const int st = plan_geometry(d, g);
    if (st != RICK_OK) return st;
    const PlanLayout L = plan_layout(d, g);
    p->grid_ok = L.grid_ok;
    p->fft_ok = L.fft_ok;
    p->gen_ok = L.gen_ok;
    p->gen = L.gen;

    int prev = 0;
    hipGetDevice(&prev);
    RICK_HIP(hipSetDevice(d.device));
    hipError_t e = hipMalloc(&p->dmem, L.bytes);
    if (e != hipSuccess) {
        hipSetDevice(prev);
        return set_error(RICK_ERR_NOMEM, "hipMalloc(%zu) failed: %s", L.bytes, hipGetErrorString(e));
    }
    p->dbytes = L.bytes;
    char *base = static_cast<char *>(p->dmem);
    p->table_d = reinterpret_cast<double *>(base + L.table);
    if (p->fft_ok && fft_needs_tmp(d.precision, g.ny)) p->tmp_plane = base + L.tmp;
    if (p->grid_ok) grid_work_carve(g, d.max_points, d.precision, base + L.work, &p->work);
    // The FP32 split-bucket accumulators and tickets start at zero (the
    // gridder leaves them zero after every call).
    if (p->grid_ok) e = hipMemset(base + L.work, 0, grid_work_bytes(g, d.max_points, d.precision));
    if (e != hipSuccess) {
        hipFree(p->dmem);
        hipSetDevice(prev);
        return set_error(RICK_ERR_DEVICE, "workspace clear failed: %s", hipGetErrorString(e));
    }

    // Host tables -> device (synchronous; plan creation is not on a hot path).
    std::vector<double> h(kMaxTable, 0.0);
    if (d.kernel != RICK_GAUSS_HI_PRECISION) kernel_table(d.kernel, d.w_support, h.data());
    // Largest per-cell weight: K[j]*K[k] <= max|K|^2, or the hi-precision
    // Gaussian's norm (w-stacking.cu:254-256, 496).
    double kmax = 0.0;
    for (int i = 0; i < g.ntable; ++i) kmax = std::max(kmax, std::fabs(h[i]));
    g.cmax = d.kernel == RICK_GAUSS_HI_PRECISION ? (1.0 / (2.0 * 1.0 * 1.0)) / kRefPi : kmax * kmax;
    g.fscale = 1.0;
    if (d.kernel != RICK_GAUSS_HI_PRECISION && kmax > 0.0)
        while (g.fscale > kmax) g.fscale *= 0.5;   // cmax / kmax = kmax
    e = hipMemcpy(p->table_d, h.data(), sizeof(double) * kMaxTable, hipMemcpyHostToDevice);
    std::vector<double> tw;
    auto put_tw = [&](int n, size_t o) {
        tw.assign(2 * (size_t)n, 0.0);
        twiddles(n, tw.data());
        if (d.precision == RICK_FP64)
            return hipMemcpy(base + o, tw.data(), 16 * (size_t)n, hipMemcpyHostToDevice);
        std::vector<float> f(tw.begin(), tw.end());
        return hipMemcpy(base + o, f.data(), 8 * (size_t)n, hipMemcpyHostToDevice);
    };
    if (e == hipSuccess) e = put_tw(g.nx, L.twx);
    if (e == hipSuccess) e = put_tw(g.ny, L.twy);
    std::vector<double> lt(g.nx), mt(g.ny);
    pixel_sines(g.nx, d.xaxistot > 0 ? d.xaxistot : g.nx, d.resolution, lt.data());
    pixel_sines(g.ny, d.yaxistot > 0 ? d.yaxistot : g.ny, d.resolution, mt.data());
    if (e == hipSuccess)
        e = hipMemcpy(base + L.l, lt.data(), sizeof(double) * g.nx, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(base + L.m, mt.data(), sizeof(double) * g.ny, hipMemcpyHostToDevice);
    if (e == hipSuccess && p->gen_ok)
        e = gen_fft_upload(&p->gen, d.precision, base + L.gen_tab, base + L.gen_work);
    hipSetDevice(prev);
    if (e != hipSuccess) {
        hipFree(p->dmem);
        return set_error(RICK_ERR_DEVICE, "table upload failed: %s", hipGetErrorString(e));
    }
    p->fft = FftPlan{g.planes, g.nx, g.ny, base + L.twx, base + L.twy};
    PhaseGeom &ph = p->phase;
    ph.planes = g.planes;
    ph.nx = g.nx;
    ph.ny = g.ny;
    ph.wmin = d.wmin;
    // phase_correction.cu:100-102
    ph.dw = (d.wmax - d.wmin) / (double)d.num_w_planes;
    ph.dwnorm = ph.dw / (d.wmax - d.wmin);
    ph.phase_on = d.phase_on;
    ph.ltab = reinterpret_cast<const double *>(base + L.l);
    ph.mtab = reinterpret_cast<const double *>(base + L.m);
    *out = p.release();
    return RICK_OK;
}

int rick_plan_describe(const rick_plan_desc *desc, unsigned int num_points, rick_plan_shape *shape)
{
    clear_error();
    if (!desc || !shape) return set_error(RICK_ERR_INVALID, "null argument");
    *shape = rick_plan_shape{};
    GridGeom g{};
    const int st = plan_geometry(*desc, g);
    if (st != RICK_OK) return st;
    if (num_points > desc->max_points)
        return set_error(RICK_ERR_INVALID, "num_points %u exceeds plan capacity %u", num_points,
                         desc->max_points);
    shape->tile_u = g.tu;
    shape->tile_v = g.tv;
    shape->rows_per_task = (int)call_rows_per_task(g, num_points);
    shape->footprint_unroll = g.smax;
    shape->by_class = tile_by_class(g);
    shape->long_tasks_first = long_tasks_first(g, desc->precision, num_points);
    shape->device_bytes = plan_layout(*desc, g).bytes;
    return RICK_OK;
}

size_t rick_plan_device_bytes(rick_plan p) { return p ? p->dbytes : 0; }

size_t rick_plan_grid_bytes(rick_plan p)
{
    if (!p) return 0;
    const size_t csz = p->d.precision == RICK_FP64 ? 16 : 8;
    return csz * (size_t)p->geom.planes * (size_t)p->geom.nx * (size_t)p->geom.ny;
}

int rick_plan_grid(rick_plan p, unsigned int n, unsigned int F, unsigned int P, const double *uu,
                   const double *vv, const double *ww, const float *vr, const float *vi,
                   const float *wt, void *grid, int accumulate, void *stream)
{
    clear_error();
    if (!p) return set_error(RICK_ERR_INVALID, "null plan");
    if (!p->grid_ok) return set_error(RICK_ERR_INVALID, "plan has no gridding capacity");
    if (n > p->d.max_points)
        return set_error(RICK_ERR_INVALID, "num_points %u exceeds plan capacity %u", n,
                         p->d.max_points);
    if (n > 0 && (F == 0 || P == 0))
        return set_error(RICK_ERR_INVALID, "freq_per_chan and polarizations must be >= 1");
    if (!grid) return set_error(RICK_ERR_INVALID, "null grid");
    if (n > 0 && (!uu || !vv || !ww || !vr || !vi || !wt))
        return set_error(RICK_ERR_INVALID, "null input array");
    RICK_HIP(hipSetDevice(p->d.device));
    RICK_HIP(launch_grid(p->geom, p->work, p->d.precision, p->table_d, n, F, P, uu, vv, ww, vr,
                         vi, wt, grid, accumulate, static_cast<hipStream_t>(stream),
                         &p->timing));
    return RICK_OK;
}

int rick_plan_fft(rick_plan p, const void *in, void *out, void *stream)
{
    clear_error();
    if (!p) return set_error(RICK_ERR_INVALID, "null plan");
    if (!p->fft_ok && !p->gen_ok)
        return set_error(RICK_ERR_UNSUPPORTED, "no FFT plan for %d x %d (axes must be >= 2)",
                         p->geom.nx, p->geom.ny);
    if (!in || !out) return set_error(RICK_ERR_INVALID, "null buffer");
    RICK_HIP(hipSetDevice(p->d.device));
    // fourier_transform.c:24
    const double norm = 1.0 / (double)((double)p->geom.nx * (double)p->geom.ny);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (p->fft_ok)
        RICK_HIP(launch_fft(p->fft, p->d.precision, in, out, p->tmp_plane, norm, s, &p->timing));
    else
        RICK_HIP(launch_fft_gen(p->gen, p->d.precision, p->geom.planes, p->geom.nx, p->geom.ny,
                                in, out, norm, s, &p->timing));
    return RICK_OK;
}

int rick_plan_phase(rick_plan p, const void *gridss, double *re, double *im, int accumulate,
                    void *stream)
{
    clear_error();
    if (!p) return set_error(RICK_ERR_INVALID, "null plan");
    if (!gridss || !re || !im) return set_error(RICK_ERR_INVALID, "null buffer");
    if (p->d.phase_on && p->geom.planes > 1 && !(p->d.wmax != p->d.wmin))
        return set_error(RICK_ERR_INVALID, "wmax == wmin: the w-plane spacing is undefined");
    RICK_HIP(hipSetDevice(p->d.device));
    RICK_HIP(launch_phase(p->phase, p->d.precision, gridss, re, im, accumulate,
                          static_cast<hipStream_t>(stream), &p->timing));
    return RICK_OK;
}

int rick_plan_profile(rick_plan p, int enable)
{
    clear_error();
    if (!p) return set_error(RICK_ERR_INVALID, "null plan");
    p->timing.on = enable != 0;
    for (auto &u : p->timing.used) u = 0;
    return RICK_OK;
}

int rick_plan_stage_times(rick_plan p, double *ms, int *launches, int n)
{
    clear_error();
    if (!p) return set_error(RICK_ERR_INVALID, "null plan");
    RICK_HIP(hipSetDevice(p->d.device));
    for (int st = 0; st < RICK_STAGE_COUNT; ++st) {
        double sum = 0.0;
        for (size_t k = 0; k < p->timing.used[st]; ++k) {
            const auto &e = p->timing.ev[st][k];
            RICK_HIP(hipEventSynchronize(e.second));
            float t = 0.0f;
            RICK_HIP(hipEventElapsedTime(&t, e.first, e.second));
            sum += t;
        }
        if (st < n) {
            if (ms) ms[st] = sum;
            if (launches) launches[st] = (int)p->timing.used[st];
        }
        p->timing.used[st] = 0;
    }
    return RICK_OK;
}

int rick_plan_grid_stats(rick_plan p, unsigned int *stats, int n)
{
    clear_error();
    if (!p || !stats) return set_error(RICK_ERR_INVALID, "null argument");
    if (!p->grid_ok) return set_error(RICK_ERR_INVALID, "plan has no gridding capacity");
    RICK_HIP(hipSetDevice(p->d.device));
    RICK_HIP(hipDeviceSynchronize());
    uint32_t meta[4] = {0, 0, 0, 0};
    RICK_HIP(hipMemcpy(meta, p->work.meta, sizeof meta, hipMemcpyDeviceToHost));
    for (int i = 0; i < n && i < 4; i++) stats[i] = meta[i];
    return RICK_OK;
}

int rick_plan_image(rick_plan p, unsigned int n, unsigned int F, unsigned int P, const double *uu,
                    const double *vv, const double *ww, const float *vr, const float *vi,
                    const float *wt, void *grid, double *re, double *im, void *stream)
{
    clear_error();
    if (!p) return set_error(RICK_ERR_INVALID, "null plan");
    if (!p->grid_ok) return set_error(RICK_ERR_INVALID, "plan has no gridding capacity");
    if (!p->fft_ok && !p->gen_ok)
        return set_error(RICK_ERR_UNSUPPORTED, "no FFT plan for %d x %d (axes must be >= 2)",
                         p->geom.nx, p->geom.ny);
    if (n > p->d.max_points)
        return set_error(RICK_ERR_INVALID, "num_points %u exceeds plan capacity %u", n,
                         p->d.max_points);
    if (n > 0 && (F == 0 || P == 0))
        return set_error(RICK_ERR_INVALID, "freq_per_chan and polarizations must be >= 1");
    if (!grid || !re || !im) return set_error(RICK_ERR_INVALID, "null buffer");
    if (n > 0 && (!uu || !vv || !ww || !vr || !vi || !wt))
        return set_error(RICK_ERR_INVALID, "null input array");
    if (p->d.phase_on && p->geom.planes > 1 && !(p->d.wmax != p->d.wmin))
        return set_error(RICK_ERR_INVALID, "wmax == wmin: the w-plane spacing is undefined");
    RICK_HIP(hipSetDevice(p->d.device));
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const double norm = 1.0 / (double)((double)p->geom.nx * (double)p->geom.ny);
    if (!p->fft_ok) {
        // Other axis lengths: the sparse chain in place where both axes are
        // smooth and rows take one pass, else a dense grid and its transform;
        // then the phase correction and plane sum.
        const bool chain = gen_chain_ok(p->gen);
        RICK_HIP(launch_grid(p->geom, p->work, p->d.precision, p->table_d, n, F, P, uu, vv, ww,
                             vr, vi, wt, grid, 0, s, &p->timing, !chain));
        if (chain) {
            RICK_HIP(launch_gen_chain(p->gen, p->d.precision, p->geom.planes, p->geom.nx,
                                      p->geom.ny, grid, norm, s, &p->timing, p->geom,
                                      p->work.offsets, p->work.rowlive, p->phase, re, im));
            return RICK_OK;
        }
        RICK_HIP(launch_fft_gen(p->gen, p->d.precision, p->geom.planes, p->geom.nx, p->geom.ny,
                                grid, grid, norm, s, &p->timing));
        RICK_HIP(launch_phase(p->phase, p->d.precision, grid, re, im, 0, s, &p->timing));
        return RICK_OK;
    }
    // Sparse grid: tiles of empty buckets are left unwritten; the row FFT
    // reads only occupied tiles (bucket offsets) and treats the rest as zero.
    // (A row of more than 256 tiles exceeds the row FFT's occupancy table;
    // such grids are cleared densely instead.)
    const bool sparse = p->geom.nx / p->geom.tu <= 256;
    RICK_HIP(launch_grid(p->geom, p->work, p->d.precision, p->table_d, n, F, P, uu, vv, ww, vr,
                         vi, wt, grid, 0, s, &p->timing, !sparse));
    RICK_HIP(launch_image_chain(p->fft, p->d.precision, grid, norm, s, &p->timing,
                                sparse ? &p->geom : nullptr, sparse ? p->work.offsets : nullptr,
                                sparse ? p->work.rowlive : nullptr, p->phase, re, im));
    return RICK_OK;
}


// ---------------------------------------------------------------------------
// Batched imaging: one plan over the group's stacked w-planes, plus the job
// tables the gridding and phase kernels read.

}  // extern "C"

struct rick_batch_s {
    rick_plan plan = nullptr;
    void *dmem = nullptr;
    size_t dbytes = 0;
    BatchJob *jobs_d = nullptr;
    PhaseJob *pjobs_d = nullptr;
    void *grid = nullptr;
    int njobs = 0;
    uint32_t vrows = 0;
    unsigned int F = 1, P = 1;
};

extern "C" {

int rick_batch_create(rick_batch *out, const rick_batch_desc *desc, const rick_batch_job *jobs,
                      int njobs)
{
    clear_error();
    if (!out || !desc || !jobs) return set_error(RICK_ERR_INVALID, "null argument");
    *out = nullptr;
    const rick_batch_desc &d = *desc;
    const int N = d.grid_size;
    if (!(is_pow2(N) && N >= 16 && N <= 8192))
        return set_error(RICK_ERR_UNSUPPORTED,
                         "batched imaging takes power-of-two grids in [16, 8192], got %d", N);
    if (njobs < 1) return set_error(RICK_ERR_INVALID, "no jobs");
    if (d.freq_per_chan == 0 || d.polarizations == 0)
        return set_error(RICK_ERR_INVALID, "freq_per_chan and polarizations must be >= 1");
    const unsigned int FP = d.freq_per_chan * d.polarizations;
    const uint64_t align = batch_row_align();
    std::vector<BatchJob> bj(njobs);
    std::vector<PhaseJob> pj(njobs);
    uint64_t vrows = 0;
    int planes = 0;
    for (int j = 0; j < njobs; ++j) {
        const rick_batch_job &J = jobs[j];
        if (J.num_w_planes < 1) return set_error(RICK_ERR_INVALID, "job %d: no w-planes", j);
        if (J.num_points > 0 && (!J.uu || !J.vv || !J.ww || !J.vis_real || !J.vis_img ||
                                 !J.weight))
            return set_error(RICK_ERR_INVALID, "job %d: null input array", j);
        if (!J.image_real || !J.image_imag)
            return set_error(RICK_ERR_INVALID, "job %d: null image", j);
        if (FP % 4 == 0 &&
            ((reinterpret_cast<uintptr_t>(J.vis_real) | reinterpret_cast<uintptr_t>(J.vis_img)) &
             15u))
            return set_error(RICK_ERR_INVALID, "job %d: visibility arrays not 16-byte aligned", j);
        if (d.phase_on && J.num_w_planes > 1 && !(J.wmax != J.wmin))
            return set_error(RICK_ERR_INVALID, "job %d: wmax == wmin", j);
        if (!(J.dw >= 0.0)) return set_error(RICK_ERR_INVALID, "job %d: negative dw", j);
        const double jdw = J.dw > 0.0 ? J.dw : 1.0 / J.num_w_planes;   // init.c:12
        bj[j] = BatchJob{J.uu, J.vv, J.ww, J.vis_real, J.vis_img, J.weight, J.num_points,
                         (uint32_t)vrows, planes, J.num_w_planes, jdw, exact_inverse(jdw)};
        // phase_correction.cu:100-102
        const double dwp = (J.wmax - J.wmin) / (double)J.num_w_planes;
        pj[j] = PhaseJob{planes, J.num_w_planes, J.wmin, dwp, dwp / (J.wmax - J.wmin),
                         d.phase_on, nullptr, nullptr, J.image_real, J.image_imag};
        vrows += ((uint64_t)J.num_points + align - 1) / align * align;
        planes += J.num_w_planes;
        if (vrows > (1ull << 30))
            return set_error(RICK_ERR_INVALID, "batch rows (padded) exceed 2^30");
    }
    rick_plan_desc pd{};
    pd.num_w_planes = planes;
    pd.grid_size_x = pd.grid_size_y = N;
    pd.kernel = d.kernel;
    pd.w_support = d.w_support;
    pd.dx = 1.0 / N;               // init.c:11
    pd.dw = 1.0;                   // each job carries its own
    pd.precision = d.precision;
    pd.max_points = (unsigned int)std::max<uint64_t>(vrows, 1);
    pd.resolution = 1.0;
    pd.wmin = 0.0;
    pd.wmax = 1.0;
    pd.phase_on = d.phase_on;
    pd.tile_u = d.tile_u;
    pd.tile_v = d.tile_v;
    pd.rows_per_task = d.rows_per_task;
    pd.device = d.device;
    pd.footprint_unroll = d.footprint_unroll;
    auto b = std::make_unique<rick_batch_s>();
    int rc = rick_plan_create(&b->plan, &pd);
    if (rc != RICK_OK) return rc;
    const size_t csz = d.precision == RICK_FP64 ? 16 : 8;
    auto al = [](size_t x) { return (x + 255) / 256 * 256; };
    size_t off = 0;
    const size_t o_jobs = off; off += al(sizeof(BatchJob) * njobs);
    const size_t o_pj = off; off += al(sizeof(PhaseJob) * njobs);
    const size_t o_lm = off; off += al(sizeof(double) * 2 * (size_t)N * njobs);
    const size_t o_grid = off; off += al(csz * (size_t)planes * N * N);
    int prev = 0;
    hipGetDevice(&prev);
    hipError_t e = hipSetDevice(d.device);
    if (e == hipSuccess) e = hipMalloc(&b->dmem, off);
    if (e != hipSuccess) {
        hipSetDevice(prev);
        rick_plan_destroy(b->plan);
        return set_error(RICK_ERR_NOMEM, "batch: hipMalloc(%zu) failed: %s", off,
                         hipGetErrorString(e));
    }
    char *base = static_cast<char *>(b->dmem);
    b->dbytes = off;
    b->jobs_d = reinterpret_cast<BatchJob *>(base + o_jobs);
    b->pjobs_d = reinterpret_cast<PhaseJob *>(base + o_pj);
    b->grid = base + o_grid;
    double *lm = reinterpret_cast<double *>(base + o_lm);
    std::vector<double> tab(2 * (size_t)N);
    for (int j = 0; j < njobs && e == hipSuccess; ++j) {
        pixel_sines(N, N, jobs[j].resolution, tab.data());          // phase_correction.cu:204-209
        pixel_sines(N, N, jobs[j].resolution, tab.data() + N);
        pj[j].ltab = lm + 2 * (size_t)N * j;
        pj[j].mtab = lm + 2 * (size_t)N * j + N;
        e = hipMemcpy(lm + 2 * (size_t)N * j, tab.data(), sizeof(double) * 2 * N,
                      hipMemcpyHostToDevice);
    }
    if (e == hipSuccess)
        e = hipMemcpy(b->jobs_d, bj.data(), sizeof(BatchJob) * njobs, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(b->pjobs_d, pj.data(), sizeof(PhaseJob) * njobs, hipMemcpyHostToDevice);
    hipSetDevice(prev);
    if (e != hipSuccess) {
        hipFree(b->dmem);
        rick_plan_destroy(b->plan);
        return set_error(RICK_ERR_DEVICE, "batch: table upload failed: %s", hipGetErrorString(e));
    }
    b->njobs = njobs;
    b->vrows = (uint32_t)vrows;
    b->F = d.freq_per_chan;
    b->P = d.polarizations;
    *out = b.release();
    return RICK_OK;
}

int rick_batch_run(rick_batch b, void *stream)
{
    clear_error();
    if (!b) return set_error(RICK_ERR_INVALID, "null batch");
    rick_plan p = b->plan;
    RICK_HIP(hipSetDevice(p->d.device));
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const bool sparse = p->geom.nx / p->geom.tu <= 256;
    RICK_HIP(launch_grid(p->geom, p->work, p->d.precision, p->table_d, b->vrows, b->F, b->P,
                         nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, b->grid, 0, s,
                         &p->timing, !sparse, b->jobs_d, b->njobs));
    const double norm = 1.0 / (double)((double)p->geom.nx * (double)p->geom.ny);
    RICK_HIP(launch_image_chain(p->fft, p->d.precision, b->grid, norm, s, &p->timing,
                                sparse ? &p->geom : nullptr, sparse ? p->work.offsets : nullptr,
                                sparse ? p->work.rowlive : nullptr, p->phase, nullptr, nullptr,
                                b->pjobs_d, b->njobs));
    return RICK_OK;
}

int rick_batch_destroy(rick_batch b)
{
    if (!b) return RICK_OK;
    int dev = 0;
    hipGetDevice(&dev);
    hipSetDevice(b->plan->d.device);
    if (b->dmem) hipFree(b->dmem);
    hipSetDevice(dev);
    rick_plan_destroy(b->plan);
    delete b;
    return RICK_OK;
}

size_t rick_batch_device_bytes(rick_batch b)
{
    return b ? b->dbytes + rick_plan_device_bytes(b->plan) : 0;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Drop-in layer: per-device context with cached plans and buffers.

namespace {

struct DevBuf {
    void *p = nullptr;
    size_t n = 0;
    int ensure(size_t bytes)
    {
        if (bytes <= n) return RICK_OK;
        if (p) hipFree(p);
        p = nullptr;
        n = 0;
        if (hipMalloc(&p, bytes) != hipSuccess)
            return set_error(RICK_ERR_NOMEM, "hipMalloc(%zu) failed", bytes);
        n = bytes;
        return RICK_OK;
    }
};

struct Ctx {
    std::mutex mu;
    int device = 0;
    hipStream_t stream = nullptr;
    rick_plan grid_plan = nullptr, phase_plan = nullptr, fft_plan = nullptr;
    DevBuf in, grid, out, img;
    // Staging between host arrays and the device: pinned pieces and their events.
    char *pinned = nullptr;
    size_t pinned_bytes = 0;
    std::vector<hipEvent_t> staged;
};

constexpr size_t kPiece = 4ull << 20;   // bytes of a staging piece
constexpr size_t kPieces = 4;           // pieces in flight
constexpr size_t kCopyShare = 256 << 10;   // least bytes of a copy per thread
// Looks (and yields) of an idle thread before it sleeps: short copies are over before a
// thread that sleeps would be back.
constexpr int kCopySpins = 4000, kLargeCopySpins = 100;
constexpr int kCopyThreads = 8;         // most threads of a copy
constexpr size_t kLarge = 256ull << 20;    // copies from here on take pieces of 32 MB

Ctx *context_for(int rank)
{
    static std::mutex mu;
    static std::vector<std::unique_ptr<Ctx>> ctxs;
    const int ndev = rick_device_count();
    if (ndev <= 0) {
        set_error(RICK_ERR_DEVICE, "no HIP device found");
        return nullptr;
    }
    const int dev = ((rank % ndev) + ndev) % ndev;
    std::lock_guard<std::mutex> lk(mu);
    if ((int)ctxs.size() < ndev) ctxs.resize(ndev);
    if (!ctxs[dev]) {
        auto c = std::make_unique<Ctx>();
        c->device = dev;
        if (hipSetDevice(dev) != hipSuccess || hipStreamCreate(&c->stream) != hipSuccess) {
            set_error(RICK_ERR_DEVICE, "cannot set up device %d", dev);
            return nullptr;
        }
        ctxs[dev] = std::move(c);
    }
    hipSetDevice(dev);
    return ctxs[dev].get();
}

bool same_plan(const rick_plan p, const rick_plan_desc &d)
{
    if (!p) return false;
    const rick_plan_desc &a = p->d;
    return a.num_w_planes == d.num_w_planes && a.grid_size_x == d.grid_size_x &&
           a.grid_size_y == d.grid_size_y && a.kernel == d.kernel && a.w_support == d.w_support &&
           a.dx == d.dx && a.dw == d.dw && a.precision == d.precision &&
           a.max_points >= d.max_points && a.resolution == d.resolution && a.wmin == d.wmin &&
           a.wmax == d.wmax && a.phase_on == d.phase_on && a.device == d.device &&
           a.tile_u == d.tile_u && a.tile_v == d.tile_v && a.rows_per_task == d.rows_per_task &&
           a.xaxistot == d.xaxistot && a.yaxistot == d.yaxistot;
}

int ensure_plan(rick_plan *slot, const rick_plan_desc &d)
{
    if (same_plan(*slot, d)) return RICK_OK;
    rick_plan_destroy(*slot);
    *slot = nullptr;
    return rick_plan_create(slot, &d);
}

// One array to or from the device, in doubles when it is added to.
struct HostCopy {
    char *dev;
    char *host;
    size_t bytes;
};
enum class Copy { to_device, to_host, add_to_host };

// Copies the arrays through pinned pieces: all threads copy (or add) their part
// of one piece while the pieces before (or after) it are on the link, which one
// thread alone cannot keep up with.  Only the calling thread makes HIP calls.
// Transfers to the device are only queued on the context's stream; the others
// are complete on return.  512^2 x 8 planes, against pageable copies to the
// device and 64 MB pieces back: wstack() 2.86 / 2.02 / 1.87 -> 2.37 / 1.39 / 1.43
// ms with 1 / 4 / 8 threads, phase_correction() 1.50 / 1.39 / 1.56 -> 1.50 / 0.96
// / 1.01, rick_fft_planes() 3.21 -> 1.74; more than 8 threads cost more to start
// than they add (16: 1.60 and 1.18 ms).  Large copies want longer pieces: wstack()
// into a grid of 8.6 GB 0.179 s (0.1790 .. 0.1792 in 12 calls with 4, 8 and 16 threads),
// with 16 MB pieces 0.183, with two of 64 MB 0.177.  Few pieces also make few commands:
// after some 500 on a stream the runtime moves it to another copy engine, and where
// that one is busy (just after gigabytes of device memory were freed) a call takes twice
// as long (0.32 s at 16 MB in every other call, 0.179 in 26 of 26 at 32 MB).  Idle
// threads sleep: 0.8 s of CPU time a call, 2.9 s while 16 of them spun.
int copy_arrays(Ctx &c, const std::vector<HostCopy> &arrays, Copy how, int nthreads)
{
    std::vector<HostCopy> pieces;
    size_t total = 0;
    for (const HostCopy &a : arrays) total += a.bytes;
    const size_t piece = total >= kLarge ? 8 * kPiece : kPiece;
    for (const HostCopy &a : arrays)
        for (size_t o = 0; o < a.bytes; o += piece)
            pieces.push_back(HostCopy{a.dev + o, a.host + o, std::min(piece, a.bytes - o)});
    const size_t n = pieces.size();
    if (how == Copy::to_device && nthreads <= 1) {
        // One thread: the runtime's own copies of pageable memory are as fast.
        for (const HostCopy &a : arrays)
            RICK_HIP(hipMemcpyAsync(a.dev, a.host, a.bytes, hipMemcpyHostToDevice, c.stream));
        return RICK_OK;
    }
    if (c.pinned_bytes < piece * kPieces) {
        if (c.pinned) {
            RICK_HIP(hipStreamSynchronize(c.stream));   // its pieces may be under way
            (void)hipHostFree(c.pinned);
            c.pinned = nullptr;
            c.pinned_bytes = 0;
        }
        void *p = nullptr;
        if (hipHostMalloc(&p, piece * kPieces, hipHostMallocDefault) != hipSuccess)
            return set_error(RICK_ERR_NOMEM, "hipHostMalloc(%zu) failed", piece * kPieces);
        c.pinned = static_cast<char *>(p);
        c.pinned_bytes = piece * kPieces;
    }
    while (c.staged.size() < kPieces) {
        hipEvent_t e = nullptr;
        RICK_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        c.staged.push_back(e);
    }
    // Pieces below `open` may be worked on; done[i] counts the finished parts of piece
    // i (a count over all pieces would let a thread that is ahead stand in for one
    // that has not started).
    std::atomic<size_t> open{how == Copy::to_device ? kPieces : 0};
    std::vector<std::atomic<int>> done(n);
    for (auto &d : done) d.store(0, std::memory_order_relaxed);
    std::atomic<int> team{0};       // threads at work, 0 until all have been started
    std::atomic<bool> stop{false};
    // A thread that has nothing to do looks again a few times, then sleeps until a
    // piece opens (helpers) or is finished (the calling thread).
    std::mutex mu;
    std::condition_variable changed;
    const int spins = total >= kLarge ? kLargeCopySpins : kCopySpins;
    auto wait_for = [&](auto &&ready) {
        for (int k = 0; k < spins; ++k) {
            if (ready()) return;
            std::this_thread::yield();
        }
        std::unique_lock<std::mutex> lk(mu);
        changed.wait(lk, ready);
    };
    auto tell = [&] {
        { std::lock_guard<std::mutex> lk(mu); }   // no waiter is between its test and its sleep
        changed.notify_all();
    };
    auto part = [&](size_t i, int t, int nt) {
        const HostCopy &p = pieces[i];
        const size_t per = ((p.bytes + nt - 1) / nt + 63) / 64 * 64;
        const size_t a = std::min(p.bytes, per * t), b = std::min(p.bytes, a + per);
        char *buf = c.pinned + (i % kPieces) * piece;
        if (how == Copy::to_device) {
            memcpy(buf + a, p.host + a, b - a);
        } else if (how == Copy::to_host) {
            memcpy(p.host + a, buf + a, b - a);
        } else {
            double *dst = reinterpret_cast<double *>(p.host + a);
            const double *src = reinterpret_cast<const double *>(buf + a);
            for (size_t q = 0; q < (b - a) / sizeof(double); ++q) dst[q] += src[q];
        }
        if (done[i].fetch_add(1, std::memory_order_acq_rel) + 1 == nt) tell();
    };
    auto helper = [&](int t) {
        wait_for([&] { return team.load(std::memory_order_acquire) > 0; });
        const int nt = team.load();
        for (size_t i = 0; i < n; ++i) {
            wait_for([&] { return open.load(std::memory_order_acquire) > i || stop.load(); });
            if (open.load(std::memory_order_acquire) <= i) return;
            part(i, t, nt);
        }
    };
    const int want = (int)std::min<size_t>(std::max(1, std::min(nthreads, kCopyThreads)),
                                           std::max<size_t>(1, total / kCopyShare));
    std::vector<std::thread> th;
    try {
        for (int t = 1; t < want; ++t) th.emplace_back(helper, t);
    } catch (const std::exception &) {
        // The threads that did start share the work.
    }
    const int nt = 1 + (int)th.size();
    team.store(nt, std::memory_order_release);
    tell();
    auto queue = [&](size_t i) {
        const HostCopy &p = pieces[i];
        char *buf = c.pinned + (i % kPieces) * piece;
        const hipError_t e =
            how == Copy::to_device
                ? hipMemcpyAsync(p.dev, buf, p.bytes, hipMemcpyHostToDevice, c.stream)
                : hipMemcpyAsync(buf, p.dev, p.bytes, hipMemcpyDeviceToHost, c.stream);
        return e != hipSuccess ? e : hipEventRecord(c.staged[i % kPieces], c.stream);
    };
    auto all_done = [&](size_t i) {
        wait_for([&] { return done[i].load(std::memory_order_acquire) >= nt; });
    };
    auto open_to = [&](size_t count) {
        open.store(count, std::memory_order_release);
        tell();
    };
    hipError_t e = hipSuccess;
    if (how != Copy::to_device)
        for (size_t i = 0; i < std::min(n, kPieces) && e == hipSuccess; ++i) e = queue(i);
    for (size_t i = 0; i < n && e == hipSuccess; ++i) {
        if (how == Copy::to_device) {
            part(i, 0, nt);
            all_done(i);
            e = queue(i);
            // The next piece to open takes the buffer of the one kPieces before it.
            if (e == hipSuccess && i + 1 >= kPieces && i + 1 < n)
                e = hipEventSynchronize(c.staged[(i + 1) % kPieces]);
            if (e == hipSuccess) open_to(std::max(kPieces, i + 2));
        } else {
            e = hipEventSynchronize(c.staged[i % kPieces]);
            if (e != hipSuccess) break;
            open_to(i + 1);
            part(i, 0, nt);
            all_done(i);
            if (i + kPieces < n) e = queue(i + kPieces);
        }
    }
    if (e != hipSuccess) {
        stop.store(true);
        tell();
    }
    for (auto &x : th) x.join();
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(c.stream);
        return set_error(RICK_ERR_DEVICE, "host copy failed: %s", hipGetErrorString(e));
    }
    return RICK_OK;
}

// Threads of a copy whose entry point names none.
int copy_threads()
{
    return std::max(1, std::min(4, (int)std::thread::hardware_concurrency() / 2));
}

void report(const char *fn)
{
    if (g_status != RICK_OK) fprintf(stderr, "[rick] %s: %s\n", fn, g_msg);
}

}  // namespace

extern "C" {

void wstack(int num_w_planes, unsigned int num_points, unsigned int freq_per_chan,
            unsigned int polarizations, double *uu, double *vv, double *ww, float *vis_real,
            float *vis_img, float *weight, double dx, double dw, int w_support, int grid_size_x,
            int grid_size_y, double *grid, int num_threads, int rank)
{
    clear_error();
    auto body = [&]() -> int {
        if (num_w_planes < 1 || grid_size_x < 1 || grid_size_y < 1 || !grid)
            return set_error(RICK_ERR_INVALID, "bad grid arguments");
        if (num_points == 0) return RICK_OK;
        if (freq_per_chan == 0 || polarizations == 0)
            return set_error(RICK_ERR_INVALID, "freq_per_chan and polarizations must be >= 1");
        Ctx *c = context_for(rank);
        if (!c) return g_status;
        std::lock_guard<std::mutex> lk(c->mu);
        rick_plan_desc d{};
        d.num_w_planes = num_w_planes;
        d.grid_size_x = grid_size_x;
        d.grid_size_y = grid_size_y;
        d.kernel = g_kernel;
        d.w_support = w_support;
        d.dx = dx;
        d.dw = dw;
        d.precision = RICK_FP64;
        d.max_points = num_points;
        d.device = c->device;
        if (c->grid_plan && same_plan(c->grid_plan, d)) d.max_points = c->grid_plan->d.max_points;
        int st = ensure_plan(&c->grid_plan, d);
        if (st != RICK_OK) return st;
        const size_t n = num_points, nv = n * freq_per_chan * polarizations,
                     nw = n * polarizations;
        auto al = [](size_t x) { return (x + 255) / 256 * 256; };
        const size_t o_u = 0, o_v = al(8 * n), o_w = o_v + al(8 * n), o_r = o_w + al(8 * n),
                     o_i = o_r + al(4 * nv), o_t = o_i + al(4 * nv), tot = o_t + al(4 * nw);
        if ((st = c->in.ensure(tot)) != RICK_OK) return st;
        const size_t gbytes = rick_plan_grid_bytes(c->grid_plan);
        if ((st = c->grid.ensure(gbytes)) != RICK_OK) return st;
        char *b = static_cast<char *>(c->in.p);
        auto host = [](const void *p) { return static_cast<char *>(const_cast<void *>(p)); };
        if ((st = copy_arrays(*c, {{b + o_u, host(uu), 8 * n}, {b + o_v, host(vv), 8 * n},
                                   {b + o_w, host(ww), 8 * n}, {b + o_r, host(vis_real), 4 * nv},
                                   {b + o_i, host(vis_img), 4 * nv},
                                   {b + o_t, host(weight), 4 * nw}},
                              Copy::to_device, num_threads)) != RICK_OK)
            return st;
        st = rick_plan_grid(c->grid_plan, num_points, freq_per_chan, polarizations,
                            reinterpret_cast<double *>(b + o_u),
                            reinterpret_cast<double *>(b + o_v),
                            reinterpret_cast<double *>(b + o_w),
                            reinterpret_cast<float *>(b + o_r), reinterpret_cast<float *>(b + o_i),
                            reinterpret_cast<float *>(b + o_t), c->grid.p, 0, c->stream);
        if (st != RICK_OK) return st;
        return copy_arrays(*c, {{static_cast<char *>(c->grid.p), reinterpret_cast<char *>(grid),
                                 gbytes}},
                           Copy::add_to_host, num_threads);
    };
    body();
    report("wstack");
}

void phase_correction(double *gridss, double *image_real, double *image_imag, int xaxis, int yaxis,
                      int num_w_planes, int xaxistot, int yaxistot, double resolution, double wmin,
                      double wmax, int num_threads, int rank)
{
    clear_error();
    auto body = [&]() -> int {
        if (!gridss || !image_real || !image_imag || xaxis < 1 || yaxis < 1 ||
            num_w_planes < 1 || xaxistot < 1 || yaxistot < 1)
            return set_error(RICK_ERR_INVALID, "bad phase_correction arguments");
        Ctx *c = context_for(rank);
        if (!c) return g_status;
        std::lock_guard<std::mutex> lk(c->mu);
        rick_plan_desc d{};
        d.num_w_planes = num_w_planes;
        d.grid_size_x = xaxis;
        d.grid_size_y = yaxis;
        d.kernel = RICK_GAUSS;
        d.w_support = 1;
        d.dx = 1.0;
        d.dw = 1.0;
        d.precision = RICK_FP64;
        d.max_points = 0;
        d.resolution = resolution;
        d.wmin = wmin;
        d.wmax = wmax;
        d.phase_on = g_phase_on;
        d.device = c->device;
        d.xaxistot = xaxistot;
        d.yaxistot = yaxistot;
        int st = ensure_plan(&c->phase_plan, d);
        if (st != RICK_OK) return st;
        const size_t gbytes = rick_plan_grid_bytes(c->phase_plan);
        const size_t npix = (size_t)xaxis * yaxis;
        if ((st = c->grid.ensure(gbytes)) != RICK_OK) return st;
        if ((st = c->img.ensure(2 * 8 * npix)) != RICK_OK) return st;
        if ((st = copy_arrays(*c, {{static_cast<char *>(c->grid.p),
                                    reinterpret_cast<char *>(gridss), gbytes}},
                              Copy::to_device, num_threads)) != RICK_OK)
            return st;
        double *re = static_cast<double *>(c->img.p), *im = re + npix;
        st = rick_plan_phase(c->phase_plan, c->grid.p, re, im, 0, c->stream);
        if (st != RICK_OK) return st;
        return copy_arrays(*c, {{reinterpret_cast<char *>(re), reinterpret_cast<char *>(image_real),
                                 8 * npix},
                                {reinterpret_cast<char *>(im), reinterpret_cast<char *>(image_imag),
                                 8 * npix}},
                           Copy::add_to_host, num_threads);
    };
    body();
    report("phase_correction");
}

void rick_fft_planes(int num_w_planes, int grid_size_x, int grid_size_y, int xaxis, int yaxis,
                     const double *grid, double *gridss, int rank)
{
    clear_error();
    auto body = [&]() -> int {
        if (!grid || !gridss || num_w_planes < 1)
            return set_error(RICK_ERR_INVALID, "bad rick_fft_planes arguments");
        if (xaxis != grid_size_x || yaxis != grid_size_y)
            return set_error(RICK_ERR_UNSUPPORTED, "multi-rank slabs are not supported");
        Ctx *c = context_for(rank);
        if (!c) return g_status;
        std::lock_guard<std::mutex> lk(c->mu);
        rick_plan_desc d{};
        d.num_w_planes = num_w_planes;
        d.grid_size_x = grid_size_x;
        d.grid_size_y = grid_size_y;
        d.kernel = RICK_GAUSS;
        d.w_support = 1;
        d.dx = 1.0;
        d.dw = 1.0;
        d.precision = RICK_FP64;
        d.device = c->device;
        int st = ensure_plan(&c->fft_plan, d);
        if (st != RICK_OK) return st;
        const size_t gbytes = rick_plan_grid_bytes(c->fft_plan);
        if ((st = c->grid.ensure(gbytes)) != RICK_OK) return st;
        if ((st = c->out.ensure(gbytes)) != RICK_OK) return st;
        if ((st = copy_arrays(*c, {{static_cast<char *>(c->grid.p),
                                    reinterpret_cast<char *>(const_cast<double *>(grid)), gbytes}},
                              Copy::to_device, copy_threads())) != RICK_OK)
            return st;
        st = rick_plan_fft(c->fft_plan, c->grid.p, c->out.p, c->stream);
        if (st != RICK_OK) return st;
        return copy_arrays(*c, {{static_cast<char *>(c->out.p), reinterpret_cast<char *>(gridss),
                                 gbytes}},
                           Copy::to_host, copy_threads());
    };
    body();
    report("rick_fft_planes");
}

}  // extern "C"
