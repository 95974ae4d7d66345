// batch_plan.cpp -- host side of the orientation-batched far field: plans (orientation
// offsets, segments, integral weights, resident workspace), the tile-shape
// autotuner, the capture-safe launch sequence and its HIP graph.
#include <hip/hip_runtime.h>

#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/abt_diff.h"
#include "batch.h"
#include "rt_internal.h"
#include "simpne.h"

namespace {

constexpr int LANES = 256;
constexpr int MAX_CHUNKS = 128;
// Segment sums kept at once: 64 bytes per bin and segment.  Orientations are run in groups whose
// segments fit; a group's last round of workgroups costs about 512 / (segments x tiles) of its time
// (0.4 % at 2 GiB).
constexpr size_t PART_BYTES = (size_t)2 << 30;
// Segment length.  The last round of workgroups idles about half a segment, 0.5 x 256 bins x len / (rate
// / 1024 slots) seconds; the segment sums cost 128 bytes per bin and segment, total / len of them, at
// ~3 TB/s.  The two are equal at len = sqrt(total x nbins x 4e-5) for ~1.2e11 beam.bins/s (the bodies run at
// 0.7e11 to 2.3e11; a factor of two either way costs under 1 % of a run), and at sqrt(total x nbins x 1.3e-5)
// for the accurate body's 0.4e11.
constexpr double SEG_RULE = 4e-5, SEG_RULE_ACCURATE = 1.3e-5;
// Below 16 beams a segment's start-up (table, bins, first records) weighs as much as its beams: 4
// orientations x 37 x 36 bins take 88, 87, 93 and 94 us a run with at least 8, 16, 24 and 32.
constexpr int64_t MIN_SEG = 16, MAX_SEG = 4096;
const int TB_CAND[3] = {8, 16, 32};
const int BPT_CAND[2] = {1, 2};

struct Shape {
    int tb = 16, bpt = 1;
    int wgs = 0;        // workgroups the chip holds at once
};

// ABI precision -> kernel variant: ABT_FP64_ACCURATE runs the accurate-phase FP64 body (3),
// ABT_FP64_FAST the restructured FP64 body (4); ABT_MIXED_GATED's tuned pass is the mixed
// body with its error scale
int kernel_prec(int precision)
{
    switch (precision) {
        case ABT_FP64_ACCURATE: return 3;
        case ABT_FP64_FAST: return 4;
        case ABT_MIXED_GATED: return 1;
        default: return precision;
    }
}
int kernel_mode(int precision) { return precision == ABT_MIXED_GATED ? abt::SWEEP_INC : abt::SWEEP_PLAIN; }

bool shape_allowed(int prec, int tb, int bpt)
{
    if (prec == ABT_FP64_ACCURATE) return tb == 16 && bpt == 1;
    if (prec == ABT_FP64_FAST) return bpt == 1 || tb <= 16;
    return true;
}

int64_t round_up(int64_t n, int64_t q) { return (n + q - 1) / q * q; }
int64_t ceil_div(int64_t n, int64_t q) { return (n + q - 1) / q; }

}  // namespace

struct abt_batch_plan {
    const abt_dev_grid* g = nullptr;
    int norient = 0, prec = 0, fast_diff = 0, cus = 256;
    std::vector<int64_t> boff, eoff;
    Shape shape;
    // the cut: segments of at most seg_len beams, orientation by orientation (beam tree, ext tree)
    int64_t seg_len = 0;
    std::vector<int32_t> seg_off;          // [2 norient + 1]
    std::vector<abt::BatchGroup> groups;
    int64_t max_segs = 0;                  // of a group: what the segment-sum buffer holds
    int nchunks = 1;                       // Mueller partial sums
    // device memory: one allocation
    void* mem = nullptr;
    size_t mem_bytes = 0;
    abt::SweepSeg* d_segs = nullptr;
    int32_t* d_seg_off = nullptr;
    double* d_w1 = nullptr;
    double* d_w2 = nullptr;
    double* d_wphi = nullptr;
    double* d_part = nullptr;        // [max_segs][8][nbins]
    double* d_pinc = nullptr;        // [max_segs][nbins] (gated)
    double* d_mpart = nullptr;       // [nchunks][16][nbins] (nchunks > 1, or gated)
    double* d_ipart = nullptr;       // [norient][ntiles][6]
    abt::GateBufs gate = {};
    // -scaling: per-orientation amplitudes, unscaled integrals, divisors; the caller's energies
    void* smem = nullptr;
    size_t smem_bytes = 0;
    abt::ScaleBufs scale = {};
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace {

int shape_for(const abt_batch_plan* p, int tb, int bpt, Shape* s)
{
    const void* k = abt_sweep_kernel(kernel_prec(p->prec), tb, bpt, kernel_mode(p->prec));
    if (!k) return abt_fail(ABT_ERR_ARG, "no batched kernel for beams_per_tile %d, bins_per_thread %d", tb, bpt);
    int n = 0;
    HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, LANES, 0));
    s->tb = tb;
    s->bpt = bpt;
    s->wgs = std::max(1, n) * p->cus;
    return 0;
}

// The segment length and table.  A rule of the plan's sizes only (not of the tile shape), so that
// every shape gives the same sums; lengths are multiples of 16, so that the mixed body's FP32 beam
// groups (of 8) are those of the uncut list.
void make_segments(abt_batch_plan* p, std::vector<abt::SweepSeg>& segs)
{
    const int n = p->norient;
    const int64_t nbins = p->g->nbins;
    const double total = (double)(p->boff[n] + p->eoff[n]);
    const double rule = p->prec == ABT_FP64_ACCURATE ? SEG_RULE_ACCURATE : SEG_RULE;
    int64_t len = std::min(MAX_SEG, std::max(MIN_SEG, round_up((int64_t)sqrt(total * (double)nbins * rule), 16)));
    // an orientation's segments fit the buffer and one launch
    const int64_t most = std::max<int64_t>(2, std::min<int64_t>(65535, (int64_t)(PART_BYTES / (64 * (size_t)nbins))));
    int64_t largest = 1;
    for (int o = 0; o < n; o++)
        largest = std::max(largest, p->boff[o + 1] - p->boff[o] + p->eoff[o + 1] - p->eoff[o]);
    len = std::max(len, most > 2 ? round_up(ceil_div(largest, most - 1), 16) : round_up(largest, 16));
    p->seg_len = len;
    p->seg_off.assign(1, 0);
    for (int o = 0; o < n; o++)
        for (int tree = 0; tree < 2; tree++) {
            const std::vector<int64_t>& off = tree ? p->eoff : p->boff;
            for (int64_t b = off[o]; b < off[o + 1]; b += len)
                segs.push_back({b, (int32_t)std::min(len, off[o + 1] - b), tree});
            p->seg_off.push_back((int32_t)segs.size());
        }
    // groups of orientations: at most `most` segments each
    p->max_segs = 1;
    for (int o = 0; o < n;) {
        int e = o + 1;
        while (e < n && p->seg_off[2 * (e + 1)] - p->seg_off[2 * o] <= most) e++;
        p->groups.push_back({o, e, p->seg_off[2 * o], p->seg_off[2 * e]});
        p->max_segs = std::max<int64_t>(p->max_segs, p->seg_off[2 * e] - p->seg_off[2 * o]);
        o = e;
    }
}

// The launches over the first `norient` orientations: groups (the plan's, cut at norient).
std::vector<abt::BatchGroup> groups_of(const abt_batch_plan* p, int norient)
{
    std::vector<abt::BatchGroup> out;
    for (const abt::BatchGroup& G : p->groups) {
        if (G.o0 >= norient) break;
        const int o1 = std::min(G.o1, norient);
        out.push_back({G.o0, o1, G.s0, p->seg_off[2 * o1]});
    }
    return out;
}

// A run of the plan's buffers in shape s.
abt::BatchRun make_run(const abt_batch_plan* p, const Shape& s, const std::vector<abt::BatchGroup>& groups,
                       int norient, const double* rb, const double* vb, const double* re, const double* ve,
                       hipStream_t st)
{
    abt::BatchRun r;
    memset(&r, 0, sizeof(r));
    r.sweep.g = p->g->d;
    r.sweep.recs[0] = rb;
    r.sweep.recs[1] = re;
    r.sweep.vrecs[0] = vb ? vb : rb;
    r.sweep.vrecs[1] = ve ? ve : re;
    r.sweep.segs = p->d_segs;
    r.sweep.part = p->d_part;
    r.sweep.ipart = p->d_pinc;
    r.sweep.fast_diff = p->fast_diff;
    r.comb.g = p->g->d;
    r.comb.part = p->d_part;
    r.comb.ipart_inc = p->d_pinc;
    r.comb.seg_off = p->d_seg_off;
    r.comb.w1 = p->d_w1;
    r.comb.w2 = p->d_w2;
    r.comb.ipart = p->d_ipart;
    r.groups = groups.data();
    r.ngroups = (int)groups.size();
    r.prec = kernel_prec(p->prec);
    r.tb = s.tb;
    r.bpt = s.bpt;
    r.norient = norient;
    r.nchunks = p->nchunks;
    r.mpart = p->d_mpart;
    r.wphi = p->d_wphi;
    r.st = st;
    return r;
}

int check_recs(const double* rb, const double* re, const abt_batch_plan* p)
{
    if (p->boff[p->norient] > 0 && !rb) return abt_fail(ABT_ERR_ARG, "batched far field: null beam records");
    if (p->eoff[p->norient] > 0 && !re) return abt_fail(ABT_ERR_ARG, "batched far field: null ext records");
    return 0;
}

void drop_graph(abt_batch_plan* p)
{
    if (p->exec) (void)hipGraphExecDestroy(p->exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    p->exec = nullptr;
    p->graph = nullptr;
}

}  // namespace

extern "C" {

int abt_batch_plan_create(const abt_dev_grid* g, int32_t norient, const int64_t* beam_off,
                          const int64_t* ext_off, int precision, int is_fast_diff, abt_batch_plan** out)
{
    if (!g || !beam_off || !ext_off || !out) return abt_fail(ABT_ERR_ARG, "abt_batch_plan_create: null argument");
    if (norient < 1) return abt_fail(ABT_ERR_ARG, "abt_batch_plan_create: need at least one orientation");
    if (precision != ABT_FP64 && precision != ABT_MIXED && precision != ABT_FP64_ACCURATE &&
        precision != ABT_FP64_FAST && precision != ABT_MIXED_GATED)
        return abt_fail(ABT_ERR_ARG, "unknown precision %d", precision);
    if (g->d.nphi < 3 || g->d.ntheta < 3)
        return abt_fail(ABT_ERR_ARG, "the phi and theta integrals (simpne) need at least 3 nodes each");
    if (beam_off[0] != 0 || ext_off[0] != 0) return abt_fail(ABT_ERR_ARG, "offsets must start at 0");
    for (int o = 0; o < norient; o++)
        if (beam_off[o + 1] < beam_off[o] || ext_off[o + 1] < ext_off[o])
            return abt_fail(ABT_ERR_ARG, "offsets must be non-decreasing (orientation %d)", o);
    int cus = 0;
    int rc = abt_ensure_device(&cus);
    if (rc) return rc;
    abt_batch_plan* p = new abt_batch_plan();
    p->g = g;
    p->norient = norient;
    p->prec = precision;
    p->fast_diff = is_fast_diff ? 1 : 0;
    p->cus = cus;
    p->boff.assign(beam_off, beam_off + norient + 1);
    p->eoff.assign(ext_off, ext_off + norient + 1);
    rc = shape_for(p, 16, 1, &p->shape);
    if (rc) { delete p; return rc; }
    std::vector<abt::SweepSeg> segs;
    make_segments(p, segs);
    const bool gated = precision == ABT_MIXED_GATED;
    const int64_t nbins = g->nbins, ntiles = ceil_div(nbins, LANES);
    int longest = 1;   // orientations of the largest group
    for (const abt::BatchGroup& G : p->groups) longest = std::max(longest, G.o1 - G.o0);
    p->nchunks = (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(4 * cus, ntiles), std::min(longest, MAX_CHUNKS)));
    const int nth = g->d.ntheta, nph = g->d.nphi;
    size_t off = 0;
    auto take = [&](size_t bytes) { size_t o = off; off += (bytes + 255) & ~(size_t)255; return o; };
    const size_t mpart_bytes = sizeof(double) * 16 * nbins * (size_t)p->nchunks;
    const size_t o_seg = take(sizeof(abt::SweepSeg) * std::max<size_t>(1, segs.size()));
    const size_t o_so = take(sizeof(int32_t) * p->seg_off.size());
    const size_t o_w1 = take(sizeof(double) * nbins);
    const size_t o_w2 = take(sizeof(double) * nbins);
    const size_t o_wp = take(sizeof(double) * nph);
    const size_t o_pt = take(sizeof(double) * 8 * nbins * (size_t)p->max_segs);
    const size_t o_mp = p->nchunks > 1 || gated ? take(mpart_bytes) : 0;
    const size_t o_ip = take(sizeof(double) * 6 * (size_t)ntiles * norient);
    const size_t o_pi = gated ? take(sizeof(double) * nbins * (size_t)p->max_segs) : 0;
    const size_t o_ep = gated ? take(sizeof(double) * nbins * (size_t)p->nchunks) : 0;
    const size_t o_est = gated ? take(sizeof(double) * nbins) : 0;
    const size_t o_fl = gated ? take(sizeof(int32_t) * nbins) : 0;
    const size_t o_li = gated ? take(sizeof(int32_t) * nbins) : 0;
    const size_t o_cn = gated ? take(sizeof(int32_t) * 64) : 0;
    if (hipMalloc(&p->mem, off) != hipSuccess) {
        delete p;
        return abt_fail(ABT_ERR_NOMEM, "batched plan: hipMalloc of %zu bytes failed", off);
    }
    p->mem_bytes = off;
    char* m = (char*)p->mem;
    p->d_segs = (abt::SweepSeg*)(m + o_seg);
    p->d_seg_off = (int32_t*)(m + o_so);
    p->d_w1 = (double*)(m + o_w1);
    p->d_w2 = (double*)(m + o_w2);
    p->d_wphi = (double*)(m + o_wp);
    p->d_part = (double*)(m + o_pt);
    if (p->nchunks > 1 || gated) p->d_mpart = (double*)(m + o_mp);
    p->d_ipart = (double*)(m + o_ip);
    if (gated) {
        p->d_pinc = (double*)(m + o_pi);
        p->gate = {(double*)(m + o_ep), (double*)(m + o_est), (int32_t*)(m + o_fl), (int32_t*)(m + o_li),
                   (int32_t*)(m + o_cn), p->d_mpart};
    }
    // integral weights: simpne over phi, then x sin(theta) / k^2 (x cos(theta)) and simpne over theta
    std::vector<double> th(nth), ph(nph), wt(nth), wp(nph), w1(nbins), w2(nbins);
    hipError_t e = hipMemcpy(th.data(), g->d.theta, sizeof(double) * nth, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(ph.data(), g->d.phi, sizeof(double) * nph, hipMemcpyDeviceToHost);
    if (e == hipSuccess) {
        abt::simpne_weights(nth, th.data(), wt.data());
        abt::simpne_weights(nph, ph.data(), wp.data());
        const double k2 = g->d.waveno * g->d.waveno;
        for (int j = 0; j < nth; j++) {
            const double st = sin(th[j]) / k2, ct = cos(th[j]);
            for (int i = 0; i < nph; i++) {
                const double w = wt[j] * st * wp[i];
                w1[i + (int64_t)nph * j] = w;
                w2[i + (int64_t)nph * j] = w * ct;
            }
        }
        e = hipMemcpy(p->d_w1, w1.data(), sizeof(double) * nbins, hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipMemcpy(p->d_w2, w2.data(), sizeof(double) * nbins, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_wphi, wp.data(), sizeof(double) * nph, hipMemcpyHostToDevice);
    if (e == hipSuccess && !segs.empty())
        e = hipMemcpy(p->d_segs, segs.data(), sizeof(abt::SweepSeg) * segs.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(p->d_seg_off, p->seg_off.data(), sizeof(int32_t) * p->seg_off.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(p->mem);
        delete p;
        return abt_fail(ABT_ERR_HIP, "batched plan upload: %s", hipGetErrorString(e));
    }
    *out = p;
    return 0;
}

int abt_batch_plan_destroy(abt_batch_plan* p)
{
    if (!p) return 0;
    drop_graph(p);
    if (p->mem) (void)hipFree(p->mem);
    if (p->smem) (void)hipFree(p->smem);
    delete p;
    return 0;
}

int abt_batch_set_scaling(abt_batch_plan* p, const double* beam_energy_out, const double* ext_energy_out)
{
    if (!p) return abt_fail(ABT_ERR_ARG, "abt_batch_set_scaling: null plan");
    if (!beam_energy_out != !ext_energy_out)
        return abt_fail(ABT_ERR_ARG, "abt_batch_set_scaling: give both energy arrays, or neither");
    if (beam_energy_out && p->prec == ABT_MIXED_GATED)
        return abt_fail(ABT_ERR_ARG, "abt_batch_set_scaling: not available for the gated mixed plan");
    int rc = abt_ensure_device(nullptr);
    if (rc) return rc;
    drop_graph(p);   // a captured graph holds the other launch sequence
    if (!beam_energy_out) {
        if (p->smem) (void)hipFree(p->smem);
        p->smem = nullptr;
        p->smem_bytes = 0;
        p->scale = {};
        return 0;
    }
    if (!p->smem) {
        const size_t nstore = (size_t)16 * p->g->nbins * p->norient;
        const size_t bytes = sizeof(double) * (nstore + 8 * (size_t)p->norient);
        void* m = nullptr;
        hipError_t e = hipMalloc(&m, bytes);
        if (e != hipSuccess)
            return abt_fail(ABT_ERR_HIP, "abt_batch_set_scaling: %zu bytes: %s", bytes, hipGetErrorString(e));
        p->smem = m;
        p->smem_bytes = bytes;
        p->scale.store = (double*)m;
        p->scale.raw = p->scale.store + nstore;
        p->scale.div = p->scale.raw + 6 * (size_t)p->norient;
    }
    p->scale.beam_energy = beam_energy_out;
    p->scale.ext_energy = ext_energy_out;
    return 0;
}

int abt_batch_set_tiles(abt_batch_plan* p, int32_t beams_per_tile, int32_t bins_per_thread)
{
    if (!p) return abt_fail(ABT_ERR_ARG, "abt_batch_set_tiles: null plan");
    Shape s;
    int rc = shape_for(p, beams_per_tile, bins_per_thread, &s);
    if (rc) return rc;
    drop_graph(p);   // a captured graph holds the old shape
    p->shape = s;
    return 0;
}

int abt_batch_get_tiles(const abt_batch_plan* p, int32_t* beams_per_tile, int32_t* bins_per_thread,
                        int32_t* chunks, int32_t* workgroups)
{
    if (!p) return abt_fail(ABT_ERR_ARG, "abt_batch_get_tiles: null plan");
    if (beams_per_tile) *beams_per_tile = p->shape.tb;
    if (bins_per_thread) *bins_per_thread = p->shape.bpt;
    if (chunks) *chunks = p->nchunks;
    if (workgroups) *workgroups = p->shape.wgs;
    return 0;
}

int abt_batch_autotune(abt_batch_plan* p, const double* recs_b, const double* vrecs_b,
                       const double* recs_e, const double* vrecs_e, int32_t sample_orient,
                       void* stream, double* ms_out)
{
    if (!p) return abt_fail(ABT_ERR_ARG, "abt_batch_autotune: null plan");
    int rc = check_recs(recs_b, recs_e, p);
    if (rc) return rc;
    rc = abt_ensure_device(nullptr);
    if (rc) return rc;
    hipStream_t st = (hipStream_t)stream;
    const int ns = std::max(1, std::min(p->norient, sample_orient > 0 ? (int)sample_orient : 32));
    const int64_t nbins = p->g->nbins;
    double* out = nullptr;
    const size_t ob = sizeof(double) * (16 * (size_t)nbins + 6 * (size_t)ns);
    HIPCHK(hipMalloc(&out, ob));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t he = hipEventCreate(&e0);
    if (he == hipSuccess) he = hipEventCreate(&e1);
    const std::vector<abt::BatchGroup> groups = groups_of(p, ns);
    float best = 1e30f;
    Shape best_s = p->shape;
    int idx = 0;
    rc = 0;
    for (int bpt : BPT_CAND) {
        for (int tb : TB_CAND) {
            if (rc || he != hipSuccess) break;
            if (!shape_allowed(p->prec, tb, bpt)) {
                if (ms_out) ms_out[idx] = 0.0;
                idx++;
                continue;
            }
            Shape s;
            rc = shape_for(p, tb, bpt, &s);
            if (rc) break;
            abt::BatchRun r = make_run(p, s, groups, ns, recs_b, vrecs_b, recs_e, vrecs_e, st);
            r.mueller = out;
            r.integrals = out + 16 * nbins;
            float ms = 0.f;
            for (int rep = 0; rep < 2 && !rc; rep++) {   // first launch warms up
                he = hipEventRecord(e0, st);
                // gated plans tune their mixed pass with its error scale
                const int le = p->prec == ABT_MIXED_GATED ? abt_launch_batch_est(&r, &p->gate) : abt_launch_batch(&r);
                if (le) rc = abt_fail(ABT_ERR_HIP, "batched launch failed: %s", hipGetErrorString((hipError_t)le));
                if (he == hipSuccess) he = hipEventRecord(e1, st);
                if (he == hipSuccess) he = hipEventSynchronize(e1);
                if (he == hipSuccess) he = hipEventElapsedTime(&ms, e0, e1);
            }
            if (ms_out) ms_out[idx] = ms;
            idx++;
            if (!rc && he == hipSuccess && ms < best) {
                best = ms;
                best_s = s;
            }
        }
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(out);
    if (rc) return rc;
    if (he != hipSuccess) return abt_fail(ABT_ERR_HIP, "autotune timing: %s", hipGetErrorString(he));
    drop_graph(p);
    p->shape = best_s;
    return 0;
}

int abt_batch_run(const abt_batch_plan* p, const double* recs_b, const double* vrecs_b,
                  const double* recs_e, const double* vrecs_e, double* dev_mueller,
                  double* dev_mueller_1d, double* dev_integrals, double* dev_ampl, void* stream)
{
    if (!p || !dev_mueller || !dev_integrals) return abt_fail(ABT_ERR_ARG, "abt_batch_run: null argument");
    int rc = check_recs(recs_b, recs_e, p);
    if (rc) return rc;
    rc = abt_ensure_device(nullptr);
    if (rc) return rc;
    abt::BatchRun r = make_run(p, p->shape, p->groups, p->norient, recs_b, vrecs_b, recs_e, vrecs_e, (hipStream_t)stream);
    r.comb.ampl_out = dev_ampl;
    r.mueller = dev_mueller;
    r.mueller_1d = dev_mueller_1d;
    r.integrals = dev_integrals;
    const int e = p->scale.beam_energy       ? abt_launch_batch_scaled(&r, &p->scale)
                  : p->prec == ABT_MIXED_GATED ? abt_launch_batch_gated(&r, &p->gate)
                                               : abt_launch_batch(&r);
    if (e) return abt_fail(ABT_ERR_HIP, "batched launch failed: %s", hipGetErrorString((hipError_t)e));
    return 0;
}

int abt_batch_capture(abt_batch_plan* p, const double* recs_b, const double* vrecs_b,
                      const double* recs_e, const double* vrecs_e, double* dev_mueller,
                      double* dev_mueller_1d, double* dev_integrals, double* dev_ampl, void* stream)
{
    if (!p) return abt_fail(ABT_ERR_ARG, "abt_batch_capture: null plan");
    if (!stream) return abt_fail(ABT_ERR_ARG, "abt_batch_capture: capture needs a non-default stream");
    int rc = abt_ensure_device(nullptr);
    if (rc) return rc;
    drop_graph(p);
    hipStream_t st = (hipStream_t)stream;
    HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    rc = abt_batch_run(p, recs_b, vrecs_b, recs_e, vrecs_e, dev_mueller, dev_mueller_1d, dev_integrals,
                       dev_ampl, stream);
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(st, &graph);
    if (rc) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
    }
    if (e != hipSuccess) return abt_fail(ABT_ERR_HIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
    hipGraphExec_t exec = nullptr;
    e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(graph);
        return abt_fail(ABT_ERR_HIP, "hipGraphInstantiate: %s", hipGetErrorString(e));
    }
    p->graph = graph;
    p->exec = exec;
    return 0;
}

int abt_batch_launch(const abt_batch_plan* p, void* stream)
{
    if (!p || !p->exec) return abt_fail(ABT_ERR_ARG, "abt_batch_launch: no captured graph (call abt_batch_capture)");
    HIPCHK(hipGraphLaunch(p->exec, (hipStream_t)stream));
    return 0;
}

int abt_batch_workspace(const abt_batch_plan* p, size_t* bytes)
{
    if (!p || !bytes) return abt_fail(ABT_ERR_ARG, "abt_batch_workspace: null argument");
    *bytes = p->mem_bytes + p->smem_bytes;
    return 0;
}

int abt_batch_gate_stats(const abt_batch_plan* p, int32_t* refined_bins, void* stream)
{
    if (!p || !refined_bins) return abt_fail(ABT_ERR_ARG, "abt_batch_gate_stats: null argument");
    if (p->prec != ABT_MIXED_GATED) {
        *refined_bins = 0;
        return 0;
    }
    hipStream_t st = (hipStream_t)stream;
    HIPCHK(hipMemcpyAsync(refined_bins, p->gate.count, sizeof(int32_t), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return 0;
}

}  // extern "C"
