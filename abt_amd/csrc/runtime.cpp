// runtime.cpp -- host side of libabt_diff.so: the C-ABI of include/abt_diff.h.
//
// Device context (lazy init, one device per process), grids resident on the
// device, host preparation of beam records (reference operation order, glibc),
// per-thread staging buffers and streams so that the host entry points are
// re-entrant, and the launch policy (beam chunking so that every launch has
// enough workgroups for 256 CUs).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <list>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/abt_diff.h"
#include "ffbody.h"
#include "frame.h"
#include "records.h"
#include "rt_internal.h"
#include "simpne.h"

extern "C" int abt_launch_far_field(const abt::DevGrid* g, const double* recs, const double* vrecs,
                                    int64_t nb, int prec, int fast_diff, int64_t per, double* out,
                                    double* work, hipStream_t st);
extern "C" int abt_launch_zero(double* out, int64_t n, hipStream_t st);
extern "C" int abt_launch_finalise(const abt::DevGrid* g, double* ab, double* ae, double* M, double* m1d,
                                   double* params, int scaling, double ebeam, double eext, hipStream_t st);
extern "C" int abt_launch_prepare(int64_t n, const double* ampl, const double* vk7,
                                  const double* prop, const double* fov, double fov_value,
                                  const int64_t* vert_off, const double* verts, double lambda,
                                  double* recs, double* vrecs, hipStream_t st);

using abt::DevGrid;

// ---------------------------------------------------------------------------
// errors
static thread_local char t_err[512];

int abt_fail(int code, const char* fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(t_err, sizeof(t_err), fmt, ap);
    va_end(ap);
    return code;
}
#define fail abt_fail


// ---------------------------------------------------------------------------
// context
namespace {

struct Context {
    std::mutex mu;
    int device = -1;
    int cus = 256;
};
Context g_ctx;

struct DevBuf {
    void* p = nullptr;
    size_t cap = 0;
};

// A device-to-host copy into ordinary memory is staged by the runtime at about 20 GB/s (4.2 MB: 213 us); through
// pinned slots, copied on while the next ones arrive, at the bus' 51 (82 us and the last slot's 14).  One aperture on
// 64,980 bins, host arrays in and out: 594 -> 225 us.
constexpr int PIN_SLOTS = 4;
constexpr size_t PIN_SLOT = (size_t)1 << 20, PIN_RING = PIN_SLOTS * PIN_SLOT;
constexpr size_t PIN_MAX = (size_t)64 << 20;   // a thread's pinned memory at most; larger inputs go unpinned
// The second stream of abt_diff_main costs about 12 us (its wait, its own copies) and hides the beam tree's way back behind
// the ext tree's sweep, whose length goes as its beams: 361 x 180 bins, us, without and with it, 1 + 1 beams 394 and
// 403, 45 + 8 455 and 449, 600 + 100 1155 and 1060.  Results that fit one slot come in one copy: 3 x 3 bins 81 -> 34,
// 181 x 45 121 -> 85.
constexpr int64_t OVERLAP_BEAMS = 8;

// per-thread staging: the host entry points may run concurrently on several threads
struct ThreadState {
    hipStream_t st = nullptr;
    DevBuf bufs[9];   // [7]: abt_far_field_dev without a workspace; [8]: the visibility entry points
    hipEvent_t ff_done = nullptr;   // the last use of bufs[7], which calls on any stream share
    std::vector<double> hrec;
    // Pinned host memory of the host entry points: PIN_SLOTS slots results come back through, then inputs.
    // One call at a time uses it (the entry points are synchronous).
    void* pin = nullptr;
    size_t pin_cap = 0;
    hipEvent_t slot_done[PIN_SLOTS] = {};
    hipStream_t back = nullptr;     // copies back while the stream's next kernel runs
    hipEvent_t first_done = nullptr;
    ThreadState* next_idle = nullptr;
};

// Every state ever made, and those of threads that have ended, for threads that begin: a program that calls from
// short-lived threads holds as much memory as it had threads at once (a state's device buffers are ordered by
// its stream and ff_done, whoever holds it).  Never destroyed: threads may end after the process's statics.
struct Registry {
    std::mutex mu;
    std::vector<ThreadState*> all;
    ThreadState* idle = nullptr;
};
Registry& registry()
{
    static Registry* r = new Registry();
    return *r;
}

struct ThreadHold {
    ThreadState* ts = nullptr;
    ~ThreadHold()
    {
        if (!ts) return;
        Registry& r = registry();
        std::lock_guard<std::mutex> lk(r.mu);
        ts->next_idle = r.idle;
        r.idle = ts;
    }
};

ThreadState& tstate()
{
    static thread_local ThreadHold h;
    if (!h.ts) {
        Registry& r = registry();
        std::lock_guard<std::mutex> lk(r.mu);
        if (r.idle) {
            h.ts = r.idle;
            r.idle = h.ts->next_idle;
        } else {
            r.all.reserve(r.all.size() + 1);
            h.ts = new ThreadState();
            r.all.push_back(h.ts);
        }
    }
    return *h.ts;
}

int ensure_device()
{
    std::lock_guard<std::mutex> lk(g_ctx.mu);
    if (g_ctx.device >= 0) {
        HIPCHK(hipSetDevice(g_ctx.device));
        return 0;
    }
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(ABT_ERR_NODEV, "no HIP device");
    HIPCHK(hipSetDevice(0));
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, 0));
    g_ctx.device = 0;
    g_ctx.cus = prop.multiProcessorCount;
    return 0;
}

// Allocations of a call on one stream while another stream is captured (by default they would invalidate that
// capture, of whatever thread): the buffers are no part of it.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

int buf_ensure(DevBuf& b, size_t bytes)
{
    if (b.cap >= bytes) return 0;
    const RelaxedCapture relaxed;
    if (b.p) HIPCHK(hipFree(b.p));
    b.p = nullptr;
    b.cap = 0;
    size_t cap = std::max(bytes, (size_t)4096);
    if (hipMalloc(&b.p, cap) != hipSuccess) {
        b.p = nullptr;
        return fail(ABT_ERR_NOMEM, "hipMalloc of %zu bytes failed", cap);
    }
    b.cap = cap;
    return 0;
}

int stream_of(ThreadState& ts)
{
    if (!ts.st) HIPCHK(hipStreamCreateWithFlags(&ts.st, hipStreamNonBlocking));
    return 0;
}

// `inputs` bytes of the thread's pinned memory, after the ring where the call copies back through it: their
// address, or null (too large, or no memory to pin), for callers to do without.
char* pin_inputs(ThreadState& ts, size_t inputs, bool with_ring = true)
{
    const size_t ring = with_ring ? PIN_RING : 0, need = ring + inputs;
    if (inputs > PIN_MAX - PIN_RING) return nullptr;
    if (ts.pin_cap < need) {
        const RelaxedCapture relaxed;
        if (ts.pin) (void)hipHostFree(ts.pin);
        ts.pin = nullptr;
        ts.pin_cap = 0;
        const size_t cap = std::min(PIN_MAX, (need + need / 4 + PIN_SLOT - 1) / PIN_SLOT * PIN_SLOT);
        if (hipHostMalloc(&ts.pin, cap, hipHostMallocDefault) != hipSuccess) {
            ts.pin = nullptr;
            (void)hipGetLastError();
            return nullptr;
        }
        ts.pin_cap = cap;
    }
    for (hipEvent_t& e : ts.slot_done)
        if (with_ring && !e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            e = nullptr;
            (void)hipGetLastError();
            return nullptr;
        }
    return (char*)ts.pin + ring;
}

// dst (host) = src (device), after what is on the stream; returns when dst holds it.  pinned: pin_inputs has
// given this call its memory.
hipError_t copy_back(ThreadState& ts, hipStream_t st, void* dst, const void* src, size_t bytes, bool pinned)
{
    if (!pinned || bytes < 65536) {   // small results take one copy either way
        hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    }
    const int64_t n = (int64_t)((bytes + PIN_SLOT - 1) / PIN_SLOT);
    const auto len = [&](int64_t k) { return std::min(PIN_SLOT, bytes - (size_t)k * PIN_SLOT); };
    const auto slot = [&](int64_t k) { return (char*)ts.pin + (size_t)(k % PIN_SLOTS) * PIN_SLOT; };
    const auto issue = [&](int64_t k) {
        hipError_t e = hipMemcpyAsync(slot(k), (const char*)src + (size_t)k * PIN_SLOT, len(k), hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? hipEventRecord(ts.slot_done[k % PIN_SLOTS], st) : e;
    };
    hipError_t e = hipSuccess;
    for (int64_t k = 0; k < std::min<int64_t>(n, PIN_SLOTS) && e == hipSuccess; k++) e = issue(k);
    for (int64_t k = 0; k < n && e == hipSuccess; k++) {
        e = hipEventSynchronize(ts.slot_done[k % PIN_SLOTS]);
        if (e != hipSuccess) break;
        memcpy((char*)dst + (size_t)k * PIN_SLOT, slot(k), len(k));
        if (k + PIN_SLOTS < n) e = issue(k + PIN_SLOTS);
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(st);   // nothing may still write the slots
    return e;
}

int check_beams(const abt_beams* b, const char* what)
{
    if (!b) return fail(ABT_ERR_ARG, "%s: null beam set", what);
    if (b->n < 0) return fail(ABT_ERR_ARG, "%s: negative beam count", what);
    if (b->n == 0) return 0;
    if (!b->ampl || !b->vk7 || !b->prop || !b->vert_off || !b->verts)
        return fail(ABT_ERR_ARG, "%s: null array", what);
    return 0;
}

int check_beams_host(const abt_beams* b, const char* what)
{
    int rc = check_beams(b, what);
    if (rc) return rc;
    if (b->n == 0) return 0;
    if (b->vert_off[0] != 0) return fail(ABT_ERR_ARG, "%s: vert_off[0] must be 0", what);
    for (int64_t i = 0; i < b->n; i++)
        if (b->vert_off[i + 1] - b->vert_off[i] < 3)
            return fail(ABT_ERR_ARG, "%s: beam %lld has fewer than 3 vertices", what, (long long)i);
    return 0;
}

// theta_i (diff_mod.f90:583-591): first theta > 1 degree (REAL*4 pi), 0-based.
// The reference leaves it undefined when there is none; here the last column.
int theta_i_of(int64_t nth, const double* th)
{
    for (int64_t j = 0; j < nth; j++)
        if (th[j] > 1 * abt::PI_R4 / 180) return (int)j;
    return (int)(nth - 1);
}

// How one orientation's beam list is cut: segments of `per` beams (a multiple of `q`), nseg of them.
struct Cut {
    int64_t per = 0;
    int nseg = 1;
    size_t work(int64_t nbins) const { return nseg > 1 ? sizeof(double) * 8 * (size_t)nbins * nseg : 0; }
};

Cut cut_into(int64_t nb, int64_t c, int64_t q)
{
    c = std::max<int64_t>(1, std::min<int64_t>(c, 32));   // the workspace is 64 B per bin per segment
    Cut k;
    k.per = std::max<int64_t>(q, ((nb + c - 1) / c + q - 1) / q * q);
    k.nseg = (int)std::max<int64_t>(1, (nb + k.per - 1) / k.per);
    return k;
}

// ~320 workgroups per CU (80 rounds at 4 resident per CU): the last round's partly filled
// CUs, and the slower forward-fallback rows, are then a small share of the launch.  Measured
// on the 200,000-aperture stress test (2533 bin tiles, mixed kernel): 4 segments run 9 % faster
// than 1, 16 a further 3 %, 32 and 64 a further 0.7 % and 1 %.  Segments keep >= 512 beams.
Cut cut_long(int64_t nbins, int64_t nb, int cus)
{
    const int64_t tiles = (nbins + 255) / 256;
    const int64_t want = ((int64_t)cus * 320 + tiles - 1) / tiles;
    return cut_into(nb, std::min<int64_t>(want, nb / 512), 32);
}

// The cut where a workspace for it is at hand, when the segments of cut_long leave the chip with few
// workgroups.  Their times differ (forward rows, branches), so the last round shrinks with their size until the
// start of a workgroup (its table, its first records) and the segment sums weigh: 24 workgroups per CU of at
// least 40 beams, and below that 8 per CU of at least 8 beams (the mixed body's group).  Measured, us, with the
// segments per list named: 3252 beams on 254 tiles of bins, plain FP64 2744 (9), 2605 (16), 2609 (24), 2583 (32),
// restructured 1412, 1283, 1238, 1230; 648 beams on them 559 (9), 538 (16), 551 (24), restructured 323, 289, 297.
Cut cut_beams(int64_t nbins, int64_t nb, int cus)
{
    const int64_t tiles = (nbins + 255) / 256;
    const Cut l = cut_long(nbins, nb, cus);
    const auto fill = [&](int64_t per_cu) { return ((int64_t)cus * per_cu + tiles - 1) / tiles; };
    const int64_t n = std::max(std::min(fill(8), nb / 8), std::min(fill(24), nb / 40));
    return n > l.nseg ? cut_into(nb, n, 8) : l;
}

}  // namespace

int abt_ensure_device(int* cus)
{
    int rc = ensure_device();
    if (!rc && cus) *cus = g_ctx.cus;
    return rc;
}

int abt_thread_staging(int slot, size_t bytes, hipStream_t* st, void** p)
{
    if (slot < 0 || slot >= 9) return fail(ABT_ERR_ARG, "staging slot %d out of range", slot);
    int rc = ensure_device();
    if (rc) return rc;
    ThreadState& ts = tstate();
    rc = stream_of(ts);
    if (!rc) rc = buf_ensure(ts.bufs[slot], bytes);
    if (rc) return rc;
    *st = ts.st;
    *p = ts.bufs[slot].p;
    return 0;
}

char* abt_thread_pinned(size_t bytes) { return pin_inputs(tstate(), bytes, false); }

// ---------------------------------------------------------------------------
// device grid

static void host_bins(int64_t nth, const double* th, int64_t nph, const double* ph, double* x,
                      double* y, double* z)
{
    // make_far_field_bins (diff_mod.f90:827-855), meshgrid layout (nphi, ntheta); the
    // sine and cosine of one angle from one sincos call, as gfortran -O3 computes them
    const double r = 1e6;
    for (int64_t j = 0; j < nth; j++)
        for (int64_t i = 0; i < nph; i++) {
            const int64_t b = i + nph * j;
            double st, ct, sp, cp;
            sincos(th[j], &st, &ct);
            sincos(ph[i], &sp, &cp);
            x[b] = r * st * cp;
            y[b] = r * st * sp;
            z[b] = -(r * ct);
        }
}

static int grid_build(int64_t nth, const double* th, int64_t nph, const double* ph,
                      const double* xs, const double* ys, const double* zs, double lambda,
                      abt_dev_grid** out)
{
    if (nth <= 0 || nph <= 0) return fail(ABT_ERR_ARG, "empty grid (%lld x %lld)", (long long)nth, (long long)nph);
    if ((double)nth * (double)nph > 2.0e9) return fail(ABT_ERR_ARG, "grid too large");
    if (!(lambda > 0)) return fail(ABT_ERR_ARG, "wavelength must be positive");
    int rc = ensure_device();
    if (rc) return rc;
    const int64_t nb = nth * nph;
    std::vector<double> h((size_t)(5 * nb + 4 * nph + 3 * nth + abt::ETAB_GRID));
    // the table first, on the allocation's own alignment: kernels read it in pairs
    double *etab = h.data(), *x = etab + abt::ETAB_GRID, *y = x + nb, *z = y + nb, *rad = z + nb, *krr = rad + nb;
    double *cp = krr + nb, *sp = cp + nph, *phv = sp + nph, *thv = phv + nph, *wph = thv + nth, *wth = wph + nph;
    abt::fill_exp_table(etab);
    memcpy(phv, ph, sizeof(double) * nph);
    memcpy(thv, th, sizeof(double) * nth);
    if (xs) {
        memcpy(x, xs, sizeof(double) * nb);
        memcpy(y, ys, sizeof(double) * nb);
        memcpy(z, zs, sizeof(double) * nb);
    } else {
        host_bins(nth, th, nph, ph, x, y, z);
    }
    const double waveno = 2.0 * abt::PI_R4 / lambda;
    const double krev = waveno / 6.283185307179586476925;
    for (int64_t b = 0; b < nb; b++) {
        const double r = sqrt(x[b] * x[b] + y[b] * y[b] + z[b] * z[b]);
        rad[b] = r;
        krr[b] = krev * r;
    }
    for (int64_t i = 0; i < nph; i++) sincos(ph[i], &sp[i], &cp[i]);
    int32_t back = 0;
    if (nph >= 3 && nth >= 3) {
        abt::simpne_weights((int)nph, ph, wph);
        abt::simpne_weights((int)nth, th, wth);
        double best = fabs(th[0] - 2 * abt::PI_R4);
        for (int64_t j = 0; j < nth; j++) {
            double s, c;
            sincos(th[j], &s, &c);
            wth[j] = wth[j] * s / (waveno * waveno);
            wth[nth + j] = wth[j] * c;
            const double d = fabs(th[j] - 2 * abt::PI_R4);
            if (d < best) { best = d; back = (int32_t)j; }
        }
    }
    abt_dev_grid* g = new abt_dev_grid();
    if (hipMalloc(&g->mem, sizeof(double) * h.size()) != hipSuccess) {
        delete g;
        return fail(ABT_ERR_NOMEM, "grid allocation failed");
    }
    if (hipMemcpy(g->mem, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(g->mem);
        delete g;
        return fail(ABT_ERR_HIP, "grid upload failed");
    }
    double* d = (double*)g->mem;
    g->d.nphi = (int32_t)nph;
    g->d.ntheta = (int32_t)nth;
    g->d.nbins = (int32_t)nb;
    g->d.theta_i = theta_i_of(nth, th);
    abt::devgrid_constants(g->d, lambda);
    if (xs) g->d.cc_far = abt::far_limit(krev, *std::min_element(rad, rad + nb));   // the caller's bins
    const auto on_device = [&](const double* p) { return d + (p - h.data()); };
    g->d.etab = on_device(etab);
    g->d.x = on_device(x);
    g->d.y = on_device(y);
    g->d.z = on_device(z);
    g->d.rad = on_device(rad);
    g->d.kr_rev = on_device(krr);
    g->d.cphi = on_device(cp);
    g->d.sphi = on_device(sp);
    g->d.phi = on_device(phv);
    g->d.theta = on_device(thv);
    g->d.wphi = on_device(wph);
    g->d.wth = on_device(wth);
    g->d.theta_back = back;
    g->nbins = nb;
    *out = g;
    return 0;
}

// ---------------------------------------------------------------------------
// Grid cache of the host entry points.  PBT calls diff_main once per orientation and,
// in -memory mode, diffraction once per beam from several OpenMP threads, always on the
// same bins: the device grid is built on the first call and kept, keyed by the exact
// contents of its inputs (angles, wavelength and, for diffraction, the caller's bin
// positions), so later calls neither rebuild nor allocate it.  Entries in use are never
// evicted; when every slot is busy a call builds a private grid and frees it.
namespace {

struct GridEntry {
    int64_t nth = 0, nph = 0;
    double lambda = 0.0;
    std::vector<double> th, ph, xyz;   // xyz empty: bins from make_far_field_bins
    abt_dev_grid* g = nullptr;
    int users = 0;
    uint64_t last = 0;
};

constexpr size_t GRID_CACHE_SLOTS = 8;
std::mutex g_grid_mu;
std::list<GridEntry> g_grids;
uint64_t g_grid_clock = 0;

bool same(const std::vector<double>& v, const double* p, int64_t n)
{
    return (int64_t)v.size() == n && (n == 0 || memcmp(v.data(), p, sizeof(double) * (size_t)n) == 0);
}

// A cached grid for these inputs (xs, ys, zs may be null), with a use held: release it
// with grid_release.  *priv is set when the grid is private to the call (cache full).
int grid_acquire(int64_t nth, const double* th, int64_t nph, const double* ph, const double* xs,
                 const double* ys, const double* zs, double lambda, abt_dev_grid** out, bool* priv)
{
    const int64_t nb = nth * nph;
    *priv = false;
    {
        std::lock_guard<std::mutex> lk(g_grid_mu);
        for (GridEntry& e : g_grids) {
            if (e.nth != nth || e.nph != nph || e.lambda != lambda) continue;
            if (!same(e.th, th, nth) || !same(e.ph, ph, nph)) continue;
            if (xs ? (e.xyz.size() != (size_t)(3 * nb) || memcmp(e.xyz.data(), xs, sizeof(double) * nb) != 0 ||
                      memcmp(e.xyz.data() + nb, ys, sizeof(double) * nb) != 0 ||
                      memcmp(e.xyz.data() + 2 * nb, zs, sizeof(double) * nb) != 0)
                   : !e.xyz.empty())
                continue;
            e.users++;
            e.last = ++g_grid_clock;
            *out = e.g;
            return 0;
        }
    }
    abt_dev_grid* g = nullptr;
    int rc = grid_build(nth, th, nph, ph, xs, ys, zs, lambda, &g);
    if (rc) return rc;
    std::lock_guard<std::mutex> lk(g_grid_mu);
    if (g_grids.size() >= GRID_CACHE_SLOTS) {
        // evict the least recently used idle entry
        auto victim = g_grids.end();
        for (auto it = g_grids.begin(); it != g_grids.end(); ++it)
            if (it->users == 0 && (victim == g_grids.end() || it->last < victim->last)) victim = it;
        if (victim == g_grids.end()) {
            *priv = true;
            *out = g;
            return 0;
        }
        abt_grid_destroy(victim->g);
        g_grids.erase(victim);
    }
    GridEntry e;
    e.nth = nth;
    e.nph = nph;
    e.lambda = lambda;
    e.th.assign(th, th + nth);
    e.ph.assign(ph, ph + nph);
    if (xs) {
        e.xyz.resize((size_t)(3 * nb));
        memcpy(e.xyz.data(), xs, sizeof(double) * nb);
        memcpy(e.xyz.data() + nb, ys, sizeof(double) * nb);
        memcpy(e.xyz.data() + 2 * nb, zs, sizeof(double) * nb);
    }
    e.g = g;
    e.users = 1;
    e.last = ++g_grid_clock;
    g_grids.push_back(std::move(e));
    *out = g;
    return 0;
}

void grid_release(abt_dev_grid* g, bool priv)
{
    if (priv) {
        abt_grid_destroy(g);
        return;
    }
    std::lock_guard<std::mutex> lk(g_grid_mu);
    for (GridEntry& e : g_grids)
        if (e.g == g) {
            e.users--;
            return;
        }
}

void grid_cache_clear()
{
    std::lock_guard<std::mutex> lk(g_grid_mu);
    for (auto it = g_grids.begin(); it != g_grids.end();) {
        if (it->users == 0) {
            abt_grid_destroy(it->g);
            it = g_grids.erase(it);
        } else {
            ++it;
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// host preparation of beam records
static void prep_range(const abt_beams* b, double fov_value, double lambda, int64_t i0, int64_t i1,
                       double* recs, double* vrecs)
{
    for (int64_t i = i0; i < i1; i++) {
        const int64_t o0 = b->vert_off[i], o1 = b->vert_off[i + 1];
        const double f = b->fov ? b->fov[i] : fov_value;
        abt::make_beam_record(b->ampl + 8 * i, b->vk7 + 3 * i, b->prop + 3 * i, f, o1 - o0,
                              b->verts + 3 * o0, lambda, o0, recs + abt::REC * i,
                              (vrecs && o1 - o0 > 3) ? vrecs + abt::VREC * o0 : nullptr);
    }
}

static void prep_host(const abt_beams* b, double fov_value, double lambda, double* recs, double* vrecs)
{
    const int64_t n = b->n;
    // 0.2 us a record against ~15 us a thread: 512 records each (3252 beams: 686 -> 250 us)
    int64_t nt = std::max(1u, std::min(std::thread::hardware_concurrency(), 16u));
    nt = std::max<int64_t>(1, std::min<int64_t>(nt, n / 512));
    const int64_t per = (n + nt - 1) / nt;
    std::vector<std::thread> th;
    int64_t i0 = 0;
    try {
        for (th.reserve((size_t)nt); i0 + per < n; i0 += per)
            th.emplace_back(prep_range, b, fov_value, lambda, i0, i0 + per, recs, vrecs);
    } catch (const std::exception&) {   // no thread to be had: the rest here
    }
    prep_range(b, fov_value, lambda, i0, n, recs, vrecs);
    for (auto& t : th) t.join();
}

static bool any_polygon(const abt_beams* b)
{
    for (int64_t i = 0; i < b->n; i++)
        if (b->vert_off[i + 1] - b->vert_off[i] > 3) return true;
    return false;
}

static size_t record_bytes(const abt_beams* b, bool poly)
{
    return sizeof(double) * (abt::REC * (size_t)b->n + (poly ? abt::VREC * (size_t)b->vert_off[b->n] : 0));
}

// Stage a host beam set on the device and run the far-field sum into dev_out.  hrec: record_bytes of host
// memory that stay until the stream is done with them (null: the thread's, for one tree at a time).
// slot: two device buffers, as hrec.
static int run_host_tree(const DevGrid& g, const abt_beams* b, bool poly, double fov_value, int prec,
                         int fast_diff, double* dev_out, ThreadState& ts, double* hrec, int slot)
{
    const int64_t n = b->n;
    hipStream_t st = ts.st;
    if (n == 0) {
        int e = abt_launch_zero(dev_out, 8 * (int64_t)g.nbins, st);
        if (e) return fail(ABT_ERR_HIP, "zero-fill launch failed: %s", hipGetErrorString((hipError_t)e));
        return 0;
    }
    const size_t bytes = record_bytes(b, poly);
    if (!hrec) {
        ts.hrec.resize(bytes / sizeof(double) + 1);
        hrec = ts.hrec.data();
    }
    prep_host(b, fov_value, g.lambda, hrec, poly ? hrec + abt::REC * n : nullptr);
    int rc = buf_ensure(ts.bufs[slot], bytes + 64);
    if (rc) return rc;
    double* drec = (double*)ts.bufs[slot].p;
    double* dvrec = poly ? drec + abt::REC * n : drec;
    HIPCHK(hipMemcpyAsync(drec, hrec, bytes, hipMemcpyHostToDevice, st));
    const Cut cut = cut_beams(g.nbins, n, g_ctx.cus);
    double* work = nullptr;
    if (cut.nseg > 1) {
        rc = buf_ensure(ts.bufs[slot + 1], cut.work(g.nbins));
        if (rc) return rc;
        work = (double*)ts.bufs[slot + 1].p;
    }
    int e = abt_launch_far_field(&g, drec, dvrec, n, prec, fast_diff, cut.per, dev_out, work, st);
    if (e) return fail(ABT_ERR_HIP, "far-field launch failed: %s", hipGetErrorString((hipError_t)e));
    return 0;
}

// ---------------------------------------------------------------------------
// C-ABI
extern "C" {

int abt_version(void) { return ABT_DIFF_ABI_VERSION; }

const char* abt_last_error(void) { return t_err; }

int abt_init(int device)
{
    std::lock_guard<std::mutex> lk(g_ctx.mu);
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(ABT_ERR_NODEV, "no HIP device");
    if (device < 0 || device >= n) return fail(ABT_ERR_ARG, "device %d out of range (%d devices)", device, n);
    HIPCHK(hipSetDevice(device));
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, device));
    if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
        return fail(ABT_ERR_NODEV, "device %d is %s, this library is built for gfx950", device, prop.gcnArchName);
    g_ctx.device = device;
    g_ctx.cus = prop.multiProcessorCount;
    return 0;
}

int abt_finalize(void)
{
    grid_cache_clear();
    Registry& r = registry();
    std::lock_guard<std::mutex> lk(r.mu);
    for (ThreadState* ts : r.all) {
        for (auto& b : ts->bufs) {
            if (b.p) (void)hipFree(b.p);
            b.p = nullptr;
            b.cap = 0;
        }
        if (ts->st) (void)hipStreamDestroy(ts->st);
        ts->st = nullptr;
        if (ts->back) (void)hipStreamDestroy(ts->back);
        ts->back = nullptr;
        for (hipEvent_t* e : {&ts->ff_done, &ts->first_done, &ts->slot_done[0], &ts->slot_done[1], &ts->slot_done[2],
                              &ts->slot_done[3]}) {
            if (*e) (void)hipEventDestroy(*e);
            *e = nullptr;
        }
        if (ts->pin) (void)hipHostFree(ts->pin);
        ts->pin = nullptr;
        ts->pin_cap = 0;
    }
    return 0;
}

int abt_make_far_field_bins(int64_t n_theta, const double* theta, int64_t n_phi, const double* phi,
                            double* x, double* y, double* z)
{
    if (n_theta <= 0 || n_phi <= 0 || !theta || !phi || !x || !y || !z)
        return fail(ABT_ERR_ARG, "abt_make_far_field_bins: bad arguments");
    host_bins(n_theta, theta, n_phi, phi, x, y, z);
    return 0;
}

int64_t abt_record_doubles(void) { return abt::REC; }
int64_t abt_vertex_record_doubles(void) { return abt::VREC; }

int abt_prepare_beams_host(const abt_beams* beams, double fov_value, double lambda, double* recs,
                           double* vrecs)
{
    int rc = check_beams_host(beams, "abt_prepare_beams_host");
    if (rc) return rc;
    if (!recs && beams->n) return fail(ABT_ERR_ARG, "abt_prepare_beams_host: null recs");
    if (!(lambda > 0)) return fail(ABT_ERR_ARG, "wavelength must be positive");
    if (!vrecs && any_polygon(beams))
        return fail(ABT_ERR_ARG, "abt_prepare_beams_host: apertures with more than 3 vertices need vrecs");
    prep_host(beams, fov_value, lambda, recs, vrecs);
    return 0;
}

int abt_prepare_beams_dev(const abt_beams* b, double fov_value, double lambda, double* dev_recs,
                          double* dev_vrecs, void* stream)
{
    int rc = check_beams(b, "abt_prepare_beams_dev");
    if (rc) return rc;
    if (!(lambda > 0)) return fail(ABT_ERR_ARG, "wavelength must be positive");
    if (b->n == 0) return 0;
    rc = ensure_device();
    if (rc) return rc;
    int e = abt_launch_prepare(b->n, b->ampl, b->vk7, b->prop, b->fov, fov_value, b->vert_off,
                               b->verts, lambda, dev_recs, dev_vrecs, (hipStream_t)stream);
    if (e) return fail(ABT_ERR_HIP, "prepare launch failed: %s", hipGetErrorString((hipError_t)e));
    return 0;
}

int abt_grid_create(const abt_grid* grid, double lambda, abt_dev_grid** out)
{
    if (!grid || !out || !grid->theta || !grid->phi) return fail(ABT_ERR_ARG, "abt_grid_create: bad arguments");
    return grid_build(grid->n_theta, grid->theta, grid->n_phi, grid->phi, nullptr, nullptr, nullptr,
                      lambda, out);
}

int abt_grid_destroy(abt_dev_grid* g)
{
    if (!g) return 0;
    if (g->mem) (void)hipFree(g->mem);
    delete g;
    return 0;
}

int64_t abt_grid_bins(const abt_dev_grid* g) { return g ? g->nbins : 0; }

size_t abt_far_field_workspace(const abt_dev_grid* g, int64_t nb, int precision)
{
    (void)precision;
    if (!g) return 0;
    if (ensure_device()) return 0;
    return cut_beams(g->nbins, nb, g_ctx.cus).work(g->nbins);
}

int abt_far_field_dev(const abt_dev_grid* g, const double* dev_recs, const double* dev_vrecs,
                      int64_t nb, int precision, int is_fast_diff, double* dev_out, void* dev_work,
                      size_t work_bytes, void* stream)
{
    if (!g || !dev_out) return fail(ABT_ERR_ARG, "abt_far_field_dev: null argument");
    if (precision != ABT_FP64 && precision != ABT_MIXED && precision != ABT_FP64_FAST)
        return fail(ABT_ERR_ARG, "unknown precision %d", precision);
    if (nb < 0) return fail(ABT_ERR_ARG, "negative beam count");
    int rc = ensure_device();
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (nb == 0) {
        int e = abt_launch_zero(dev_out, 8 * (int64_t)g->nbins, st);
        if (e) return fail(ABT_ERR_HIP, "zero-fill launch failed: %s", hipGetErrorString((hipError_t)e));
        return 0;
    }
    if (!dev_recs) return fail(ABT_ERR_ARG, "abt_far_field_dev: null records");
    // The long segments where a caller's workspace is too small for the finer cut's.  A graph outlives the call, so
    // a captured call without a workspace has no buffer to take: the thread's may be replaced, and is
    // ordered between eager calls only.  It runs in one segment, which needs none (3252 beams on 64,980 bins, plain
    // FP64: 6.7 ms against 2.7 with a workspace; on 519,120 bins 24.8 against 20.6).
    Cut cut = cut_beams(g->nbins, nb, g_ctx.cus);
    void* work = dev_work;
    ThreadState* shared = nullptr;
    if (work) {
        if (work_bytes < cut.work(g->nbins)) cut = cut_long(g->nbins, nb, g_ctx.cus);
        if (work_bytes < cut.work(g->nbins))
            return fail(ABT_ERR_ARG, "workspace of %zu bytes is smaller than the %zu needed", work_bytes, cut.work(g->nbins));
    } else if (cut.nseg > 1) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (st) HIPCHK(hipStreamIsCapturing(st, &cs));   // (the null stream cannot be captured)
        if (cs != hipStreamCaptureStatusNone) {
            cut = cut_into(nb, 1, 8);
        } else {
            ThreadState& ts = tstate();
            rc = buf_ensure(ts.bufs[7], cut.work(g->nbins));
            if (rc) return rc;
            work = ts.bufs[7].p;
            // a call of this thread on another stream may still be reading the buffer
            if (!ts.ff_done) HIPCHK(hipEventCreateWithFlags(&ts.ff_done, hipEventDisableTiming));
            else HIPCHK(hipStreamWaitEvent(st, ts.ff_done, 0));
            shared = &ts;
        }
    }
    int e = abt_launch_far_field(&g->d, dev_recs, dev_vrecs ? dev_vrecs : dev_recs, nb, precision,
                                 is_fast_diff, cut.per, dev_out, (double*)work, st);
    if (shared) HIPCHK(hipEventRecord(shared->ff_done, st));
    if (e) return fail(ABT_ERR_HIP, "far-field launch failed: %s", hipGetErrorString((hipError_t)e));
    return 0;
}

int abt_far_field_incoherent_dev(const abt_dev_grid* g, const double* dev_recs,
                                 const double* dev_vrecs, int64_t nb, int is_fast_diff,
                                 double* dev_intensity, void* stream)
{
    if (!g || !dev_intensity) return fail(ABT_ERR_ARG, "abt_far_field_incoherent_dev: null argument");
    if (nb < 0) return fail(ABT_ERR_ARG, "negative beam count");
    int rc = ensure_device();
    if (rc) return rc;
    if (nb == 0) {
        int e = abt_launch_zero(dev_intensity, g->nbins, (hipStream_t)stream);
        if (e) return fail(ABT_ERR_HIP, "zero-fill launch failed: %s", hipGetErrorString((hipError_t)e));
        return 0;
    }
    if (!dev_recs) return fail(ABT_ERR_ARG, "abt_far_field_incoherent_dev: null records");
    int e = abt_launch_far_field(&g->d, dev_recs, dev_vrecs ? dev_vrecs : dev_recs, nb, 2, is_fast_diff, nb,
                                 dev_intensity, nullptr, (hipStream_t)stream);
    if (e) return fail(ABT_ERR_HIP, "far-field launch failed: %s", hipGetErrorString((hipError_t)e));
    return 0;
}

int abt_diff_main(const abt_grid* grid, double lambda, int is_fast_diff, const abt_beams* beams,
                  const abt_beams* ext, int precision, double* ampl_far_beam, double* ampl_far_ext_diff)
{
    const bool want_b = ampl_far_beam != nullptr, want_e = ampl_far_ext_diff != nullptr;
    if (!grid || (!want_b && !want_e)) return fail(ABT_ERR_ARG, "abt_diff_main: null argument");
    if (precision != ABT_FP64 && precision != ABT_MIXED && precision != ABT_FP64_FAST)
        return fail(ABT_ERR_ARG, "unknown precision %d", precision);
    int rc = want_b ? check_beams_host(beams, "abt_diff_main(beams)") : 0;
    if (rc) return rc;
    rc = want_e ? check_beams_host(ext, "abt_diff_main(ext)") : 0;
    if (rc) return rc;
    if (!grid->theta || !grid->phi) return fail(ABT_ERR_ARG, "abt_diff_main: null angles");
    abt_dev_grid* g = nullptr;
    bool priv = false;
    rc = grid_acquire(grid->n_theta, grid->theta, grid->n_phi, grid->phi, nullptr, nullptr, nullptr, lambda, &g,
                      &priv);
    if (rc) return rc;
    ThreadState& ts = tstate();
    rc = stream_of(ts);
    const size_t ob = sizeof(double) * 8 * (size_t)g->nbins;
    if (!rc) rc = buf_ensure(ts.bufs[0], 2 * ob);
    if (!rc) {
        double* d0 = (double*)ts.bufs[0].p;
        double* d1 = d0 + 8 * g->nbins;
        // Both trees' records in pinned memory: the ext tree's are prepared while the beam tree's kernel
        // runs, and with OVERLAP_BEAMS and more of them the beam tree's result comes back meanwhile.
        const bool pb = want_b && any_polygon(beams), pe = want_e && any_polygon(ext);
        const size_t rb = want_b ? record_bytes(beams, pb) : 0, re = want_e ? record_bytes(ext, pe) : 0;
        char* pin = pin_inputs(ts, rb + re);
        const auto hip = [&](hipError_t e, const char* what) {
            if (e != hipSuccess && !rc) rc = fail(ABT_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
        };
        const bool both = want_b && want_e && pin, one_copy = both && 2 * ob <= PIN_SLOT;
        const bool apart = both && !one_copy && ext->n >= OVERLAP_BEAMS;
        if (apart && !ts.back) hip(hipStreamCreateWithFlags(&ts.back, hipStreamNonBlocking), "stream");
        if (apart && !rc && !ts.first_done) hip(hipEventCreateWithFlags(&ts.first_done, hipEventDisableTiming), "event");
        if (!rc && want_b)
            rc = run_host_tree(g->d, beams, pb, 0.0, precision, is_fast_diff, d0, ts, (double*)pin, 1);
        if (!rc && apart) {
            hip(hipEventRecord(ts.first_done, ts.st), "event");
            if (!rc) hip(hipStreamWaitEvent(ts.back, ts.first_done, 0), "event");
        } else if (!rc && want_b && want_e && !pin) {
            // the ext tree's staging must not overwrite the beam tree's still in flight
            hip(hipStreamSynchronize(ts.st), "stream sync");
        }
        // ext-diff beams: fov = pi/2 (diff_mod.f90:797)
        if (!rc && want_e) {
            abt_beams e2 = *ext;
            e2.fov = nullptr;
            rc = run_host_tree(g->d, &e2, pe, abt::PI_R4 / 2.0, precision, is_fast_diff, d1, ts,
                               pin ? (double*)(pin + rb) : nullptr, both ? 3 : 1);
        }
        if (!rc && one_copy) {   // the two results lie side by side
            hip(hipMemcpyAsync(ts.pin, d0, 2 * ob, hipMemcpyDeviceToHost, ts.st), "copy-back");
            if (!rc) hip(hipStreamSynchronize(ts.st), "copy-back");
            if (!rc) {
                memcpy(ampl_far_beam, ts.pin, ob);
                memcpy(ampl_far_ext_diff, (char*)ts.pin + ob, ob);
            }
        } else {
            if (!rc && want_b) hip(copy_back(ts, apart ? ts.back : ts.st, ampl_far_beam, d0, ob, pin != nullptr), "copy-back");
            if (!rc && want_e) hip(copy_back(ts, ts.st, ampl_far_ext_diff, d1, ob, pin != nullptr), "copy-back");
        }
        if (rc) {   // nothing may still read the staging
            (void)hipStreamSynchronize(ts.st);
            if (ts.back) (void)hipStreamSynchronize(ts.back);
        }
    }
    grid_release(g, priv);
    return rc;
}

int abt_diffraction(int64_t n_phi, int64_t n_theta, const double* xfar, const double* yfar,
                    const double* zfar, double lambda, const double* phi_vals,
                    const double* theta_vals, int is_fast_diff, const double* ampl,
                    const double* vk7, const double* prop, double fov, int64_t nv,
                    const double* verts, int precision, double* amplC)
{
    if (!xfar || !yfar || !zfar || !phi_vals || !theta_vals || !ampl || !vk7 || !prop || !verts || !amplC)
        return fail(ABT_ERR_ARG, "abt_diffraction: null argument");
    if (nv < 3) return fail(ABT_ERR_ARG, "abt_diffraction: aperture needs at least 3 vertices");
    if (precision != ABT_FP64 && precision != ABT_MIXED && precision != ABT_FP64_FAST)
        return fail(ABT_ERR_ARG, "unknown precision %d", precision);
    abt_dev_grid* g = nullptr;
    bool priv = false;
    int rc = grid_acquire(n_theta, theta_vals, n_phi, phi_vals, xfar, yfar, zfar, lambda, &g, &priv);
    if (rc) return rc;
    ThreadState& ts = tstate();
    rc = stream_of(ts);
    const size_t ob = sizeof(double) * 8 * (size_t)g->nbins;
    if (!rc) rc = buf_ensure(ts.bufs[0], ob);
    if (!rc) {
        int64_t off[2] = {0, nv};
        abt_beams b = {1, ampl, vk7, prop, &fov, off, verts};
        char* pin = pin_inputs(ts, record_bytes(&b, nv > 3));
        rc = run_host_tree(g->d, &b, nv > 3, fov, precision, is_fast_diff, (double*)ts.bufs[0].p, ts, (double*)pin, 1);
        if (!rc) {
            hipError_t e = copy_back(ts, ts.st, amplC, ts.bufs[0].p, ob, pin != nullptr);
            if (e != hipSuccess) rc = fail(ABT_ERR_HIP, "copy-back: %s", hipGetErrorString(e));
        } else {
            (void)hipStreamSynchronize(ts.st);
        }
    }
    grid_release(g, priv);
    return rc;
}

size_t abt_finalise_workspace(const abt_dev_grid* g)
{
    if (!g) return 0;
    return sizeof(double) * (8 * (size_t)g->nbins + 3 * (size_t)g->d.ntheta);
}

int abt_finalise_dev(const abt_dev_grid* g, double* ab, double* ae, int scaling, double ebeam,
                     double eext, double* dev_mueller, double* dev_m1d, double* dev_params,
                     void* dev_work, size_t work_bytes, void* stream)
{
    if (!g || !ab || !ae || !dev_mueller || !dev_m1d || !dev_params)
        return fail(ABT_ERR_ARG, "abt_finalise_dev: null argument");
    if (g->d.nphi < 3 || g->d.ntheta < 3)
        return fail(ABT_ERR_ARG, "finalise needs at least 3 theta and 3 phi values (simpne)");
    if (scaling && !(ebeam > 0 && eext > 0))
        return fail(ABT_ERR_ARG, "energy scaling needs positive beam and ext energies");
    int rc = ensure_device();
    if (rc) return rc;
    // (the epilogue keeps nothing between its kernels but its outputs; a caller's workspace is only checked)
    const size_t need = abt_finalise_workspace(g);
    if (dev_work && work_bytes < need)
        return fail(ABT_ERR_ARG, "finalise workspace of %zu bytes is smaller than %zu", work_bytes, need);
    int e = abt_launch_finalise(&g->d, ab, ae, dev_mueller, dev_m1d, dev_params, scaling, ebeam, eext,
                                (hipStream_t)stream);
    if (e) return fail(ABT_ERR_HIP, "finalise launch failed: %s", hipGetErrorString((hipError_t)e));
    return 0;
}

int abt_finalise(const abt_grid* grid, double lambda, double* ampl_far_beam, double* ampl_far_ext_diff,
                 int scaling, double beam_energy_out, double ext_energy_out, double* mueller,
                 double* mueller_beam, double* mueller_ext, double* mueller_1d,
                 double* mueller_1d_beam, double* mueller_1d_ext, double* params)
{
    if (!grid || !ampl_far_beam || !ampl_far_ext_diff || !grid->theta || !grid->phi)
        return fail(ABT_ERR_ARG, "abt_finalise: null argument");
    abt_dev_grid* g = nullptr;
    bool priv = false;
    int rc = grid_acquire(grid->n_theta, grid->theta, grid->n_phi, grid->phi, nullptr, nullptr, nullptr, lambda, &g,
                          &priv);
    if (rc) return rc;
    ThreadState& ts = tstate();
    rc = stream_of(ts);
    const int64_t nb = g->nbins, nth = g->d.ntheta;
    const size_t ob = sizeof(double) * 8 * nb;
    const size_t mb = sizeof(double) * 16 * nb, m1b = sizeof(double) * 16 * nth;
    if (!rc) rc = buf_ensure(ts.bufs[0], 2 * ob + 3 * mb + 3 * m1b + 16 * sizeof(double));
    if (!rc) {
        double* dab = (double*)ts.bufs[0].p;
        double* dae = dab + 8 * nb;
        double* dM = dae + 8 * nb;
        double* dm1 = dM + 48 * nb;
        double* dpar = dm1 + 48 * nth;
        hipStream_t st = ts.st;
        hipError_t e = hipMemcpyAsync(dab, ampl_far_beam, ob, hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipMemcpyAsync(dae, ampl_far_ext_diff, ob, hipMemcpyHostToDevice, st);
        if (e != hipSuccess) rc = fail(ABT_ERR_HIP, "upload: %s", hipGetErrorString(e));
        if (!rc) rc = abt_finalise_dev(g, dab, dae, scaling, beam_energy_out, ext_energy_out, dM, dm1,
                                       dpar, nullptr, 0, st);
        if (!rc) {
            struct { void* h; const void* d; size_t n; } cp[] = {
                {ampl_far_beam, dab, ob}, {ampl_far_ext_diff, dae, ob},
                {mueller, dM, mb}, {mueller_beam, dM + 16 * nb, mb}, {mueller_ext, dM + 32 * nb, mb},
                {mueller_1d, dm1, m1b}, {mueller_1d_beam, dm1 + 16 * nth, m1b},
                {mueller_1d_ext, dm1 + 32 * nth, m1b}, {params, dpar, 9 * sizeof(double)}};
            for (auto& c : cp) {
                if (!c.h) continue;
                e = hipMemcpyAsync(c.h, c.d, c.n, hipMemcpyDeviceToHost, st);
                if (e != hipSuccess) break;
            }
            if (e == hipSuccess) e = hipStreamSynchronize(st);
            if (e != hipSuccess) rc = fail(ABT_ERR_HIP, "copy-back: %s", hipGetErrorString(e));
        }
    }
    grid_release(g, priv);
    return rc;
}

}  // extern "C"
