// visibility.hip -- the facets a propagating beam illuminates (the near-field
// tracer's visibility step), bit-identical to find_vis_int / find_vis_ext /
// find_vis_inc (beam_loop_mod.f90:2037-2609).
//
// The reference, per beam: 16 boxes on a 4 x 4 grid over the x-y extent of
// the vertices (beam_aligned_bounding_boxes, :2668-2743); each facet's box is
// the one whose midpoint is nearest its midpoint (f3), and a facet is a
// candidate blocker in every box nearest to one of its first three vertices
// (f4, f5).  A tested facet m then scans the candidates j of its box in facet
// order: j must lie in front (mid_z(m) <= mid_z(j)) and cover m's midpoint in
// projection (edge checks); the first non-beam blocker of another aperture
// ends the scan, beam facets record the nearest one (id_beam, dist_beam).
//
// Here, for many beams at once:
//   k_vis_setup   one workgroup per beam: x-y extents (block min/max), the boxes, then per facet its box,
//                 candidate mask, cull and shadow flags and initial outputs; field_in -> mapping
//                 (last position wins, as the reference's sequential store); per box the ascending
//                 candidate list and the ascending list of tested facets (each wave owns a run of facets
//                 and writes after the waves before it, so list order is facet order);
//   k_vis_main    one wave per 64 tested facets of one box: every lane of the
//                 wave scans the same candidate list in facet order, so a candidate is wave-uniform: its
//                 list entry comes through scalar loads and its projected vertices as broadcasts
//                 from LDS, where the workgroup keeps its beam's vertices; a lane
//                 stops at its blocker, the wave when all lanes have stopped.
// Triangles seen from the side on which no midpoint can pass their edge checks are left out (see faces_away).
// All arithmetic is the reference's FP64 operations with contraction off and
// comparisons in the same sense; min/max reductions are exact, so results do
// not depend on the decomposition.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <limits.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include "../../include/abt_vis.h"
#include "rt_internal.h"

namespace abt {
namespace vis {

constexpr int NB = 16;                                // 4 x 4 boxes
constexpr int BLK = 256;
constexpr int SETUP = 256, SETUP_FEW = 1024;          // threads of k_vis_setup: many beams, few
constexpr int WAVE = 64;
constexpr int XCDS = 8;                               // dies, which workgroups go round
constexpr int MW = 4;                                 // waves of a k_vis_main workgroup
constexpr int OFFS = 2 * (NB + 1) + 2;                // per-beam list offsets (padded)
constexpr int UNR = 4;                                // candidates evaluated together in the scan
constexpr int64_t STAGE_NV = 3584;                    // vertices of a beam kept in LDS, at most (56 KB of 64)
constexpr int64_t BEAM_CHUNK = 65535;                 // beams per launch (grid.y)
constexpr double FAC = 1.100000023841858;             // fac = 1.1, a REAL*4 literal (:2679)
constexpr double C001 = 0.009999999776482582;         // 0.01, a REAL*4 literal

// One entry of a candidate list.
struct __align__(32) Cand {
    double z;        // depth of the facet's midpoint
    int j;           // facet
    int v[3];        // its first vertices; v[0] < 0: not a triangle; v[1] < 0: faces away (only counted)
    int ap, map;     // aperture, position in field_in (0: not a beam facet)
};

// A wave-uniform entry through scalar loads: the lists are not written while a scan runs, which the constant
// address space says (the scan's own stores of its results would otherwise rule it out).
__device__ __forceinline__ Cand load_scalar(const Cand* p)
{
    typedef int Words __attribute__((ext_vector_type(8)));
    static_assert(sizeof(Words) == sizeof(Cand), "an entry is 32 bytes");
    return __builtin_bit_cast(Cand, *(const __attribute__((address_space(4))) Words*)(uintptr_t)p);
}

struct Work {
    uint32_t* fbits;    // [nbeam][nf] bits 0-15: candidate blocker in box k; F_BOX, F_TESTED, F_AWAY
    int32_t* mapping;   // [nbeam][nf] 1-based position in field_in (the last), 0: not a beam facet
    int32_t* offs;      // [nbeam][OFFS] candidate-list offsets [0..NB], tested-list offsets [NB+1..2NB+1]
    Cand* cand;         // [nbeam][3 nf]
    int32_t* mlist;     // [nbeam][nf]
    int64_t nvref;      // f_off[nf]
    int64_t b0;         // first beam of this launch
    int nb, parts;      // beams of this launch; workgroups of k_vis_main per beam
    int keep_all;       // lists for a counted scan: the facets that face away too
};
constexpr uint32_t F_BOX = 16, F_TESTED = 1u << 20, F_AWAY = 1u << 21;   // F_BOX: shift of the tested facet's box

__device__ __forceinline__ int64_t clampi(int64_t i, int64_t n) { return i < 0 ? 0 : (i >= n ? n - 1 : i); }

// minloc over the box midpoints of sqrt((bx - px)**2 + (by - py)**2), first minimum
// (beam_loop_mod.f90:2087-2093), box k = 4 i + j at (bx[i], by[j]).
// The square root is monotonic, so the smallest distance is the root of the smallest
// squared distance; a box before it ties with it only if its squared distance rounds to the same
// root, which needs d2 <= dmin (1 + 2^-51).  Rounded sums are monotonic too: the smallest d2 is that of
// the smallest dx^2 and dy^2, and if neither the second smallest of each with the smallest of the
// other comes within the limit, no other box does.  The rest (ties, points that are not finite) scan all
// boxes as the reference does; finite: the boxes are.
// lx, ly: bx, by in memory, for the rare path's rolled loop.
__device__ __forceinline__ int nearest_box(const double* bx, const double* by, const double* lx, const double* ly,
                                           bool finite, double px, double py)
{
#pragma clang fp contract(off)
    double m[2], n[2];   // smallest and second smallest squared offset in x, y
    int k[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        double d[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const double o = (c ? by[i] : bx[i]) - (c ? py : px);
            d[i] = o * o;
        }
        k[c] = d[1] < d[0] ? 1 : 0;
        m[c] = fmin(d[0], d[1]);
        n[c] = fmax(d[0], d[1]);
#pragma unroll
        for (int i = 2; i < 4; i++) {
            k[c] = d[i] < m[c] ? i : k[c];
            n[c] = fmin(n[c], fmax(m[c], d[i]));
            m[c] = fmin(m[c], d[i]);
        }
    }
    const double dmin = m[0] + m[1], lim = dmin + ldexp(dmin, -49);
    if (finite && n[0] + m[1] > lim && m[0] + n[1] > lim) return 4 * k[0] + k[1];
    double best = 0.0;
    int kb = 0;
#pragma unroll 1
    for (int q = 0; q < NB; q++) {
        const double dx = lx[q >> 2] - px, dy = ly[q & 3] - py;
        const double d = sqrt(dx * dx + dy * dy);
        if (q == 0 || d < best) {
            best = d;
            kb = q;
        }
    }
    return kb;
}

// Whether no midpoint can pass the edge checks of this triangle, rounding included.  The exact checks of the
// three edges, C_e = (m - x_e) x (x_e+1 - x_e), add up to minus twice the signed area whatever m is, so one of them
// is at least a third of it when the area is negative (positive for find_vis_ext, whose checks have
// the other sign): outside that edge.  A computed check is within 4 u (|m_x - x_e| |e_y| + |m_y - y_e| |e_x|)
// of C_e, u = 1.1e-16, as is the computed area of its own; the extents of vertices and midpoints together, ex
// and ey, bound the offsets.  64 u covers the factors 3, 4 and their sum four times over.  A midpoint that is NaN
// is outside no edge: with one among them, or one infinite, ex or ey is infinite and no triangle faces away.
__device__ __forceinline__ bool faces_away(int mode, double x0, double y0, double x1, double y1, double x2, double y2,
                                           double ex, double ey)
{
    const double ax = x1 - x0, ay = y1 - y0, bx = x2 - x0, by = y2 - y0;
    const double area2 = ax * by - ay * bx;
    const double lx = fmax(fabs(ax), fmax(fabs(bx), fabs(x2 - x1))), ly = fmax(fabs(ay), fmax(fabs(by), fabs(y2 - y1)));
    const double tol = 7.2e-15 * (ex * ly + ey * lx);
    return mode == ABT_VIS_EXT ? area2 > tol : area2 < -tol;
}

__device__ __forceinline__ double wave_min(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const double w = __shfl_xor(v, o, 64);
        v = w < v ? w : v;
    }
    return v;
}
__device__ __forceinline__ double wave_max(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const double w = __shfl_xor(v, o, 64);
        v = w > v ? w : v;
    }
    return v;
}

__device__ __forceinline__ int lanes_below(unsigned long long m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// ---------------------------------------------------------------------------
// Everything before the scan, one workgroup per beam.  Bound by memory where there are many beams (31 bytes a
// facet of initial outputs, 32 a list entry, 64 read), by the latency of its steps for one beam.  As four
// kernels (boxes, facets, map, lists) with each facet's box and mask in memory between them, sixteen
// distances a search and four barriers a block of 256 facets in the list building, 2048 beams x 2112
// facets took 256 us; here 184.  One beam: 49 us and two more launches; here 30.
// STAGE: the beam's projected vertices are kept in LDS (nv <= STAGE_NV): their gathers, 64 lines each,
// otherwise fill the CU's address unit.
template <bool STAGE>
__global__ __launch_bounds__(SETUP_FEW) void k_vis_setup(abt_vis_batch a, Work w)
{
#pragma clang fp contract(off)
    constexpr int NQ = 2 * NB;   // q < NB: candidate list of box q; q >= NB: tested list of box q - NB
    constexpr int NWMAX = SETUP_FEW / WAVE;
    extern __shared__ double2 sxy[];
    __shared__ double red[NWMAX][12];
    __shared__ double sbx[4], sby[4], sext[6];
    __shared__ int s_cnt[NWMAX][NQ];
    const int64_t b = w.b0 + blockIdx.x;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wv = tid / WAVE, nt = blockDim.x, nw = nt / WAVE;
    const int64_t nf = a.nf;
    const double* x = a.v + 3 * a.nv * b;
    const double* y = x + a.nv;
    const double* fmid = a.f_mid + 3 * nf * b;
    {
        // extents: the vertices', the illuminating facets', the midpoints'
        double r[12];
#pragma unroll
        for (int q = 0; q < 12; q += 2) {
            r[q] = INFINITY;
            r[q + 1] = -INFINITY;
        }
        const auto grow = [&](int q, double px, double py) {
            r[q] = px < r[q] ? px : r[q];
            r[q + 1] = px > r[q + 1] ? px : r[q + 1];
            r[q + 2] = py < r[q + 2] ? py : r[q + 2];
            r[q + 3] = py > r[q + 3] ? py : r[q + 3];
        };
        for (int64_t i = tid; i < a.nv; i += nt) {
            const double px = x[i], py = y[i];
            if (STAGE) sxy[i] = make_double2(px, py);
            grow(0, px, py);
        }
        if (a.mode != ABT_VIS_INC) {
            const int64_t e0 = a.in_off[b], e1 = a.in_off[b + 1];
            for (int64_t e = e0 + tid; e < e1; e += nt) {
                const int64_t fi = clampi(a.field_in[e] - 1, nf);
                for (int64_t k = a.f_off[fi]; k < a.f_off[fi + 1]; k++) {
                    const int64_t vk = clampi(a.f_vi[k] - 1, a.nv);
                    grow(4, x[vk], y[vk]);
                }
            }
        }
        for (int64_t i = tid; i < nf; i += nt) {
            const double px = fmid[3 * i], py = fmid[3 * i + 1];
            grow(8, px, py);
            if (px != px || py != py) r[9] = INFINITY;   // outside no edge: see faces_away
        }
#pragma unroll
        for (int q = 0; q < 12; q++) r[q] = (q & 1) ? wave_max(r[q]) : wave_min(r[q]);
        if (lane == 0) {
#pragma unroll
            for (int q = 0; q < 12; q++) red[wv][q] = r[q];
        }
        __syncthreads();
        if (tid < 12) {
            double v = red[0][tid];
            for (int k = 1; k < nw; k++) {
                const double u = red[k][tid];
                v = (tid & 1) ? (u > v ? u : v) : (u < v ? u : v);
            }
            red[0][tid] = v;
        }
        __syncthreads();
        if (tid < 8) {
            // box corners fac * (min + (max - min) / 4 * (i - 1)) (:2711-2720), box k = 4 (i-1) + (j-1)
            // with corners (i, j), (i, j+1), (i+1, j+1), (i+1, j) summed in that order, / 4 (:2732-2740,
            // compute_geometry_midpoints misc_submod.f90:199-209)
            const int c = tid >> 2, i = (tid & 3) + 1;
            const double lo = red[0][2 * c], hi = red[0][2 * c + 1];
            const double p0 = FAC * (lo + (hi - lo) / 4.0 * (double)(i - 1));
            const double p1 = FAC * (lo + (hi - lo) / 4.0 * (double)i);
            if (c == 0)
                sbx[i - 1] = ((((0.0 + p0) + p0) + p1) + p1) / 4.0;
            else
                sby[i - 1] = ((((0.0 + p0) + p1) + p1) + p0) / 4.0;
        } else if (tid < 14) {
            const int q = tid - 8;   // the illuminating facets' extents, then the widths of vertices and midpoints
            const double* e = red[0];
            sext[q] = q < 4 ? e[4 + q] : fmax(e[2 * q - 7], e[2 * q + 1]) - fmin(e[2 * q - 8], e[2 * q]);
        }
        __syncthreads();
    }
    double bx[4], by[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        bx[k] = sbx[k];
        by[k] = sby[k];
    }
    bool finite = true;
#pragma unroll
    for (int k = 0; k < 4; k++) finite = finite && isfinite(bx[k]) && isfinite(by[k]);
    const double ex = sext[4], ey = sext[5];
    const auto vertex = [&](int64_t q) { return clampi(a.f_vi[q < w.nvref ? q : w.nvref - 1] - 1, a.nv); };
    const auto at = [&](int v) { return STAGE ? sxy[v] : make_double2(x[v], y[v]); };
    // facets: each wave a run of whole 64s, in wave order
    const int64_t run = ((nf + WAVE - 1) / WAVE + nw - 1) / nw * WAVE;
    const int64_t i0 = run * wv, i1 = i0 + run < nf ? i0 + run : nf;
    uint32_t* fbits = w.fbits + nf * b;
    int cnt = 0;   // lane q: entries of list q
    for (int64_t base = i0; base < i1; base += WAVE) {
        const int64_t i = base + lane;
        uint32_t bits = 0;
        if (i < i1) {
            const double mx = fmid[3 * i], my = fmid[3 * i + 1];
            const double nz = a.f_nz[nf * b + i];
            const int64_t api = a.f_ap[i];
            const double apn = a.ap_nz[a.na * b + clampi(api - 1, a.na)];
            const int64_t o0 = a.f_off[i];
            const bool tri = a.f_off[i + 1] - o0 == 3;
            const int v0 = (int)vertex(o0), v1 = (int)vertex(o0 + 1), v2 = (int)vertex(o0 + 2);
            bool vis = true;
            if (a.mode != ABT_VIS_INC) {   // midpoint outside the beam's extent (:2145-2155)
                if (mx < sext[0]) vis = false;
                else if (mx > sext[1]) vis = false;
                else if (my < sext[2]) vis = false;
                else if (my > sext[3]) vis = false;
            }
            const bool shad = a.mode == ABT_VIS_INT ? nz >= 0 : nz <= 0;                 // :2158, :2370, :2543
            const bool down = a.mode == ABT_VIS_INT ? apn > -C001 : apn < C001;          // :2165, :2377, :2547
            const bool tested = vis && !down;
            const int64_t o = nf * b + i;
            a.in_beam[o] = (a.mode == ABT_VIS_INC && !down) ? 1 : 0;
            if (a.is_vis) a.is_vis[o] = tested ? 1 : 0;
            a.dist_beam[o] = 0.0;
            a.id_beam[o] = 0;
            a.is_shad[o] = shad ? 1 : 0;
            w.mapping[o] = 0;
            // Neighbours agree, so a wave mostly skips the search of the midpoint's box or the vertices'.
            // The incident beam's blockers face up (:2553).
            bool away = false;
            if (tri) {
                const double2 p0 = at(v0), p1 = at(v1), p2 = at(v2);
                away = faces_away(a.mode, p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, ex, ey);
            }
            if (tested) bits = F_TESTED | (uint32_t)nearest_box(bx, by, sbx, sby, finite, mx, my) << F_BOX;
            if (!(a.mode == ABT_VIS_INC && nz < C001) && (w.keep_all || !away)) {
                if (away) bits |= F_AWAY;
#pragma unroll 1
                for (int q = 0; q < 3; q++) {
                    const double2 p = at(q == 0 ? v0 : (q == 1 ? v1 : v2));
                    bits |= 1u << nearest_box(bx, by, sbx, sby, finite, p.x, p.y);
                }
            }
            fbits[i] = bits;
        }
        const uint32_t box = bits & F_TESTED ? (bits >> F_BOX) & (NB - 1) : NB;
#pragma unroll 4
        for (int q = 0; q < NB; q++) {
            const int n = __popcll(__ballot((bits >> q) & 1u)), t = __popcll(__ballot(box == (uint32_t)q));
            cnt += lane == q ? n : (lane == NB + q ? t : 0);
        }
    }
    if (lane < NQ) s_cnt[wv][lane] = cnt;
    __syncthreads();   // (orders the zeroed mapping before the atomics too)
    int32_t* mapping = w.mapping + nf * b;
    if (a.mode != ABT_VIS_INC) {
        const int64_t e0 = a.in_off[b], e1 = a.in_off[b + 1];
        for (int64_t e = e0 + tid; e < e1; e += nt) {
            const int64_t fi = a.field_in[e] - 1;
            if (fi < 0 || fi >= nf) continue;
            atomicMax(mapping + fi, (int)(e - e0 + 1));
        }
    }
    // where list q of this wave's run starts (lane q): the lists before it, the waves before this one
    int pos = 0;
    {
        int tot = 0, before = 0;
        if (lane < NQ)
            for (int k = 0; k < nw; k++) {
                const int n = s_cnt[k][lane];
                before += k < wv ? n : 0;
                tot += n;
            }
        int end = tot;   // inclusive prefix within each 16 lists
#pragma unroll
        for (int o = 1; o < NB; o <<= 1) {
            const int u = __shfl_up(end, o, NB);
            end += (lane & (NB - 1)) >= o ? u : 0;
        }
        pos = end - tot + before;
        if (wv == 0 && lane < NQ) {
            int32_t* offs = w.offs + (int64_t)OFFS * b + (lane / NB) * (NB + 1);
            offs[lane & (NB - 1)] = end - tot;
            if ((lane & (NB - 1)) == NB - 1) offs[NB] = end;
        }
    }
    __syncthreads();   // the mapping is complete
    Cand* cand = w.cand + 3 * nf * b;
    int32_t* mlist = w.mlist + nf * b;
    for (int64_t base = i0; base < i1; base += WAVE) {
        const int64_t i = base + lane;
        const uint32_t bits = i < i1 ? fbits[i] : 0u;
        const uint32_t box = bits & F_TESTED ? (bits >> F_BOX) & (NB - 1) : NB;
        Cand c;
        if (bits & 0xffffu) {
            const int64_t o0 = a.f_off[i];
            c.z = fmid[3 * i + 2];
            c.j = (int)i;
#pragma unroll
            for (int q = 0; q < 3; q++) c.v[q] = (int)vertex(o0 + q);
            if (a.f_off[i + 1] - o0 != 3) c.v[0] |= INT_MIN;
            if (bits & F_AWAY) c.v[1] |= INT_MIN;
            c.ap = (int)a.f_ap[i];
            // written by atomics in L2, past this CU's cache
            c.map = __hip_atomic_load(mapping + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        for (int q = 0; q < NQ; q++) {
            const bool in = q < NB ? (bits >> q) & 1u : box == (uint32_t)(q - NB);
            const unsigned long long bal = __ballot(in);
            if (!bal) continue;
            const int p = __builtin_amdgcn_readlane(pos, q) + lanes_below(bal);
            if (in) {
                if (q < NB) cand[p] = c;
                else mlist[p] = (int32_t)i;
            }
            pos += lane == q ? __popcll(bal) : 0;
        }
    }
}

// ---------------------------------------------------------------------------
// The scan.  int, ext: each wave one unit (box, 64-facet slice of the box's tested list).  inc: the candidates'
// effects are ORs and ANDs, in any order, so the workgroup's waves share one unit and take a part of its
// candidates each, which a single incident beam (48 units on the whole chip) needs.
// Bound by VALU issue and by the length of a beam's last units.  Nothing is gathered per lane: a tile of
// candidates gathered lane by lane (13 loads of 64 lines each: entry, facet, vertices) kept the CU's
// address unit busy for as long as the scan of the tile took, and waited for three loads in a row.  The
// workgroup's waves take its units as they come free; a workgroup per few units, each wave with one,
// left half the waves without work.  2048 beams x 2112 facets: 536 -> 324 us (half of the scan from leaving out
// the candidates that face away); one incident beam 45 -> 10 us.  STAGE: vertices in LDS; beyond STAGE_NV
// from memory.
template <int MODE, bool COUNT, bool STAGE>
__global__ __launch_bounds__(MW * WAVE, COUNT ? 4 : 8) void k_vis_main(abt_vis_batch a, Work w)
{
#pragma clang fp contract(off)
    constexpr bool SHARE = MODE == ABT_VIS_INC;
    extern __shared__ double2 sxy[];
    __shared__ int s_res[SHARE ? MW : 1][WAVE];
    __shared__ int s_next;
    __shared__ uint64_t s_work[COUNT ? MW : 1][2];
    // workgroups go round the XCDs: all of a beam's on one, next to each other, the one its set-up ran on
    const int k8 = blockIdx.x / XCDS, bi = k8 / w.parts * XCDS + blockIdx.x % XCDS, part = k8 % w.parts;
    if (bi >= w.nb) return;
    const int64_t b = w.b0 + bi;
    const int lane = threadIdx.x & (WAVE - 1), wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int64_t nf = a.nf;
    const int32_t* offs = w.offs + (int64_t)OFFS * b;
    // lane k: the end of box k's units (64-facet slices of its tested list) among the beam's
    int ends = 0;
    if (lane < NB) ends = (offs[NB + 2 + lane] - offs[NB + 1 + lane] + WAVE - 1) / WAVE;
#pragma unroll
    for (int o = 1; o < NB; o <<= 1) {
        const int e = __shfl_up(ends, o, NB);
        ends += lane >= o ? e : 0;
    }
    const int total = __builtin_amdgcn_readlane(ends, NB - 1);
    if (part >= total) return;   // no unit for the workgroup
    const double* vx = a.v + 3 * a.nv * b;
    const double* vy = vx + a.nv;
    if (STAGE) {
        for (int i = threadIdx.x; i < (int)a.nv; i += MW * WAVE) sxy[i] = make_double2(vx[i], vy[i]);
    }
    if (threadIdx.x == 0) s_next = 0;
    __syncthreads();
    const auto at = [&](int v) { return STAGE ? sxy[v] : make_double2(vx[v], vy[v]); };
    // units part, part + parts, ...: taken by the waves as they come free, or (SHARE) by all waves together
    uint64_t npair = 0, nedge = 0;
    for (int n = 0;; n++) {
        if (!SHARE) {
            int t = 0;
            if (lane == 0) t = atomicAdd(&s_next, 1);
            n = __builtin_amdgcn_readfirstlane(t);
        }
        const int u = part + n * w.parts;
        if (u >= total) break;
        const int bb = __popcll(__ballot(lane < NB && ends <= u));
        const int t = u - (bb > 0 ? __builtin_amdgcn_readlane(ends, bb - 1) : 0);
        const int mi = offs[NB + 1 + bb] + t * WAVE + lane;
        const bool has = mi < offs[NB + 2 + bb];
        const int m = has ? w.mlist[nf * b + mi] : 0;
        const double* mid = a.f_mid + 3 * nf * b + 3 * (int64_t)m;
        const double mx = mid[0], my = mid[1], mz = mid[2];
        const int apm = (int)a.f_ap[m];
        const Cand* cand = w.cand + 3 * nf * b;
        bool done = !has;
        bool vis = true, inb = MODE == ABT_VIS_INC, shad = false;
        int32_t idb = 0;
        double dist = 0.0, zbest = 0.0;
        // edge k from vertex k to k+1 (the last back to the first): edge_norm1 = y_{k+1} - y_k,
        // edge_norm2 = -x_{k+1} + x_k, offset (mx - x_k, my - y_k) (:2149-2162)
        const auto outside = [&](double2 p, double2 q) {
#pragma clang fp contract(off)
            const double en2 = -q.x + p.x, en1 = q.y - p.y;
            const double vb1 = mx - p.x, vb2 = my - p.y;
            const double chk = MODE == ABT_VIS_EXT ? -vb1 * en1 - vb2 * en2 : vb1 * en1 + vb2 * en2;
            return chk > 0;
        };
        int c0 = offs[bb], c1 = offs[bb + 1];
        if (SHARE) {
            const int n = c1 - c0;
            c1 = c0 + (int)((int64_t)n * (wv + 1) / MW);
            c0 = c0 + (int)((int64_t)n * wv / MW);
        }
        // UNR candidates at a time: their depth and edge tests are independent of the scan state,
        // so they are evaluated together (their loads and FP64 chains overlap); the
        // reference's order-dependent rules are then applied to them in candidate order.
        for (int c = c0; c < c1; c += UNR) {
            if (__all(done)) break;
            bool pr[UNR], fr[UNR], hit[UNR];
            Cand e[UNR];
#pragma unroll
            for (int q = 0; q < UNR; q++) e[q] = load_scalar(cand + min(c + q, c1 - 1));
            bool poly = false;
#pragma unroll
            for (int q = 0; q < UNR; q++) {
                // (past the end the last candidate comes again, which changes nothing but the counts)
                pr[q] = (!COUNT || c + q < c1) && e[q].j != m;
                fr[q] = pr[q] && !(mz > e[q].z);                         // blocker not behind m
                const double2 p0 = at(e[q].v[0] & INT_MAX), p1 = at(e[q].v[1] & INT_MAX), p2 = at(e[q].v[2]);
                const bool o0 = outside(p0, p1), o1 = outside(p1, p2), o2 = outside(p2, p0);
                hit[q] = fr[q] && !(o0 || o1 || o2);
                poly = poly || e[q].v[0] < 0;
            }
            if (poly) {   // uniform
#pragma unroll
                for (int q = 0; q < UNR; q++) {
                    if (e[q].v[0] >= 0) continue;
                    const int64_t o0 = a.f_off[e[q].j];
                    const int nv = (int)(a.f_off[e[q].j + 1] - o0);
                    const double2 p0 = at(e[q].v[0] & INT_MAX);
                    double2 p = p0;
                    bool within = true;
                    for (int k = 1; k <= nv; k++) {
                        const int64_t o = o0 + k < w.nvref ? o0 + k : w.nvref - 1;
                        const double2 n = k == nv ? p0 : at((int)clampi(a.f_vi[o] - 1, a.nv));
                        within = within && !outside(p, n);
                        p = n;
                    }
                    hit[q] = fr[q] && within;
                }
            }
#pragma unroll
            for (int q = 0; q < UNR; q++) {
                if (!COUNT && !__any(hit[q] && !done)) continue;
                if (done) break;
                if (COUNT) {
                    npair += pr[q] ? 1 : 0;
                    nedge += fr[q] ? (uint64_t)(e[q].v[0] >= 0 ? 3 : a.f_off[e[q].j + 1] - a.f_off[e[q].j]) : 0;
                }
                if (!hit[q]) continue;
                if (MODE == ABT_VIS_INC) {                                // :2573-2580
                    if (apm == e[q].ap) shad = true;
                    else {
                        vis = false;
                        inb = false;
                    }
                    continue;
                }
                if (e[q].map > 0) {                                       // a beam facet: keep the nearest (:2166-2180)
                    if (!inb || e[q].z < zbest) {
                        inb = true;
                        idb = e[q].map;
                        dist = e[q].z - mz;
                        zbest = e[q].z;
                    }
                } else {                                                  // a blocker (:2181-2197)
                    if (apm == e[q].ap) continue;
                    if (inb && e[q].z > zbest) continue;
                    vis = false;
                    inb = false;
                    done = true;
                }
            }
        }
        if (SHARE) {   // blocked (2) and shadowed (1) by any of the waves' candidates
            s_res[wv][lane] = (inb ? 0 : 2) | (shad ? 1 : 0);
            __syncthreads();
            int r = 0;
#pragma unroll
            for (int k = 0; k < MW; k++) r |= s_res[k][lane];
            __syncthreads();
            inb = vis = !(r & 2);
            shad = r & 1;
        }
        if (has && (!SHARE || wv == 0)) {
            const int64_t o = nf * b + m;
            a.in_beam[o] = inb ? 1 : 0;
            if (a.is_vis) a.is_vis[o] = vis ? 1 : 0;
            if (MODE == ABT_VIS_INC) {                                    // :2597-2602
                if (shad) a.is_shad[o] = 1;
                if (inb) {
                    a.dist_beam[o] = a.beam_mid_z[b] - mz;
                    a.id_beam[o] = 1;
                }
            } else {
                a.dist_beam[o] = dist;
                a.id_beam[o] = idb;
            }
        }
    }
    if (COUNT) {   // one atomic of two lanes a workgroup: one a wave and counter queued for longer than the scan took
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            npair += __shfl_xor(npair, o, 64);
            nedge += __shfl_xor(nedge, o, 64);
        }
        if (lane == 0) {
            s_work[wv][0] = npair;
            s_work[wv][1] = nedge;
        }
        __syncthreads();
        if (threadIdx.x < 2) {
            uint64_t n = 0;
#pragma unroll
            for (int k = 0; k < MW; k++) n += s_work[k][threadIdx.x];
            if (n) atomicAdd(a.counts + threadIdx.x, (unsigned long long)n);
        }
    }
}

// ---------------------------------------------------------------------------
// rotate (beam_loop_mod.f90:1467-1526) applied to many beams: vertices, facet normals,
// midpoints and aperture normals each multiplied by the beam's rotation, every element as
// ((r_i1 p_1 + r_i2 p_2) + r_i3 p_3) like the reference's matmul (contraction off).
__device__ __forceinline__ double rot_row(const double* R, int i, double px, double py, double pz)
{
#pragma clang fp contract(off)
    double a = R[3 * i] * px;
    a = a + R[3 * i + 1] * py;
    a = a + R[3 * i + 2] * pz;
    return a;
}

__global__ __launch_bounds__(BLK) void k_vis_rotate(int64_t b0, const double* __restrict__ rot, int64_t nv,
                                                    const double* __restrict__ v0, int64_t nf,
                                                    const double* __restrict__ mid0, const double* __restrict__ n0,
                                                    int64_t na, const double* __restrict__ apn0,
                                                    double* __restrict__ v, double* __restrict__ mid,
                                                    double* __restrict__ nz, double* __restrict__ ap_nz)
{
    const int64_t b = b0 + blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * BLK + threadIdx.x;
    double R[9];
#pragma unroll
    for (int k = 0; k < 9; k++) R[k] = rot[9 * b + k];
    if (i < nv) {
        const double x = v0[i], y = v0[nv + i], z = v0[2 * nv + i];
        double* o = v + 3 * nv * b;
        o[i] = rot_row(R, 0, x, y, z);
        o[nv + i] = rot_row(R, 1, x, y, z);
        o[2 * nv + i] = rot_row(R, 2, x, y, z);
    }
    if (i < nf) {
        const double* p = mid0 + 3 * i;
        double* o = mid + 3 * nf * b + 3 * i;
        o[0] = rot_row(R, 0, p[0], p[1], p[2]);
        o[1] = rot_row(R, 1, p[0], p[1], p[2]);
        o[2] = rot_row(R, 2, p[0], p[1], p[2]);
        const double* q = n0 + 3 * i;
        nz[nf * b + i] = rot_row(R, 2, q[0], q[1], q[2]);
    }
    if (i < na) {
        const double* q = apn0 + 3 * i;
        ap_nz[na * b + i] = rot_row(R, 2, q[0], q[1], q[2]);
    }
}

}  // namespace vis
}  // namespace abt

// ---------------------------------------------------------------------------
// host side
namespace {

using abt::vis::Work;

constexpr size_t ALIGN = 256;
size_t up(size_t n) { return (n + ALIGN - 1) / ALIGN * ALIGN; }

struct Layout {
    size_t fbits, mapping, offs, cand, mlist, total;
};

Layout layout(int64_t nbeam, int64_t nf, int64_t nvref)
{
    Layout L;
    size_t o = 0;
    const size_t nb = (size_t)nbeam, f = (size_t)nf;
    L.fbits = o;   o += up(nb * f * 4);
    L.mapping = o; o += up(nb * f * 4);
    L.offs = o;    o += up(nb * abt::vis::OFFS * 4);
    L.cand = o;    o += up(nb * 3 * f * sizeof(abt::vis::Cand));
    L.mlist = o;   o += up(nb * f * 4);
    L.total = o;
    return L;
}

int launch_all(const abt_vis_batch& a, int64_t nvref, char* ws, int cus, hipStream_t st)
{
    using namespace abt::vis;
    const Layout L = layout(a.nbeam, a.nf, nvref);
    Work w;
    w.fbits = (uint32_t*)(ws + L.fbits);
    w.mapping = (int32_t*)(ws + L.mapping);
    w.offs = (int32_t*)(ws + L.offs);
    w.cand = (Cand*)(ws + L.cand);
    w.mlist = (int32_t*)(ws + L.mlist);
    w.nvref = nvref;
    // A scan alone that counts sets up once more: the set-up before it need not have listed the facets that face
    // away, which are half of a scan's entries (4096 beams x 2112 facets in phases: scan 1.08 -> 0.59 ms).
    w.keep_all = a.counts != nullptr;
    const bool stage = a.nv <= STAGE_NV;
    const size_t lds = stage ? sizeof(double2) * (size_t)a.nv : 0;
    // 64-facet slices of the tested lists, at most
    const int64_t slices = (a.nf + WAVE - 1) / WAVE + NB;
    const bool setup = a.phases != 2 || a.counts, scan = a.phases != 1;
    for (int64_t b0 = 0; b0 < a.nbeam; b0 += BEAM_CHUNK) {
        const unsigned nb = (unsigned)std::min<int64_t>(BEAM_CHUNK, a.nbeam - b0);
        w.b0 = b0;
        if (setup) {
            // with fewer beams than CUs a workgroup may as well be large
            const unsigned nt = nb < 256 && a.nf > SETUP ? SETUP_FEW : SETUP;
            if (stage) hipLaunchKernelGGL(k_vis_setup<true>, dim3(nb), dim3(nt), lds, st, a, w);
            else hipLaunchKernelGGL(k_vis_setup<false>, dim3(nb), dim3(nt), 0, st, a, w);
        }
        if (!scan) continue;
        // As many workgroups a beam as there are units for, up to twice the chip's (8 per CU at 8 waves per SIMD): a
        // beam's last unit then holds fewer waves up (2048 beams: 0.63, 0.57, 0.57 ms a batch with 1, 2, 4).
        const int64_t most = a.mode == ABT_VIS_INC ? slices : (slices + MW - 1) / MW;
        w.nb = (int)nb;
        w.parts = (int)std::max<int64_t>(1, std::min<int64_t>(most, (16 * cus + nb - 1) / nb));
        const dim3 g((nb + XCDS - 1) / XCDS * XCDS * (unsigned)w.parts), wg(MW * WAVE);
#define VM(M)                                                                                            \
    do {                                                                                                 \
        if (a.counts && stage) hipLaunchKernelGGL((k_vis_main<M, true, true>), g, wg, lds, st, a, w);    \
        else if (a.counts) hipLaunchKernelGGL((k_vis_main<M, true, false>), g, wg, 0, st, a, w);         \
        else if (stage) hipLaunchKernelGGL((k_vis_main<M, false, true>), g, wg, lds, st, a, w);          \
        else hipLaunchKernelGGL((k_vis_main<M, false, false>), g, wg, 0, st, a, w);                      \
    } while (0)
        if (a.mode == ABT_VIS_INT) VM(ABT_VIS_INT);
        else if (a.mode == ABT_VIS_EXT) VM(ABT_VIS_EXT);
        else VM(ABT_VIS_INC);
#undef VM
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return abt_fail(ABT_ERR_HIP, "visibility launch failed: %s", hipGetErrorString(e));
    return 0;
}

int check_batch(const abt_vis_batch* a)
{
    if (!a) return abt_fail(ABT_ERR_ARG, "abt_find_vis_dev: null batch");
    if (a->mode != ABT_VIS_INT && a->mode != ABT_VIS_EXT && a->mode != ABT_VIS_INC)
        return abt_fail(ABT_ERR_ARG, "unknown visibility mode %d", a->mode);
    if (a->nbeam < 0 || a->nf < 1 || a->nv < 1 || a->na < 1)
        return abt_fail(ABT_ERR_ARG, "visibility: need nbeam >= 0, nf, nv, na >= 1");
    if (a->nf >= (1LL << 31) / 3) return abt_fail(ABT_ERR_ARG, "visibility: too many facets (%lld)", (long long)a->nf);
    if (a->nv >= (1LL << 31)) return abt_fail(ABT_ERR_ARG, "visibility: too many vertices (%lld)", (long long)a->nv);
    if (!a->f_off || !a->f_vi || !a->f_ap || !a->v || !a->f_mid || !a->f_nz || !a->ap_nz || !a->in_off ||
        !a->in_beam || !a->dist_beam || !a->id_beam || !a->is_shad)
        return abt_fail(ABT_ERR_ARG, "visibility: null array");
    if (a->mode != ABT_VIS_INC && !a->field_in) return abt_fail(ABT_ERR_ARG, "visibility: null field_in");
    if (a->mode == ABT_VIS_INC && !a->beam_mid_z) return abt_fail(ABT_ERR_ARG, "find_vis_inc needs beam_mid_z");
    if (a->phases < 0 || a->phases > 3) return abt_fail(ABT_ERR_ARG, "visibility: phases must be 0..3");
    return 0;
}

}  // namespace

extern "C" size_t abt_find_vis_workspace(int64_t nbeam, int64_t nf, int64_t nvref)
{
    if (nbeam < 0 || nf < 0 || nvref < 0) return 0;
    return layout(nbeam, nf, nvref).total;
}

extern "C" int abt_find_vis_dev(const abt_vis_batch* a, int64_t nvref, void* workspace, size_t bytes,
                                void* stream)
{
    int rc = check_batch(a);
    if (rc) return rc;
    if (a->nbeam == 0) return 0;
    if (nvref < 3 * a->nf) return abt_fail(ABT_ERR_ARG, "visibility: nvref %lld < 3 nf", (long long)nvref);
    if (nvref >= (1LL << 31)) return abt_fail(ABT_ERR_ARG, "visibility: too many vertex references");
    const size_t need = abt_find_vis_workspace(a->nbeam, a->nf, nvref);
    if (!workspace || bytes < need)
        return abt_fail(ABT_ERR_ARG, "visibility workspace of %zu bytes is smaller than %zu", bytes, need);
    if ((uintptr_t)workspace % ALIGN) return abt_fail(ABT_ERR_ARG, "visibility workspace is not 256-byte aligned");
    int cus = 0;
    rc = abt_ensure_device(&cus);
    if (rc) return rc;
    return launch_all(*a, nvref, (char*)workspace, cus, (hipStream_t)stream);
}

extern "C" int abt_find_vis(int mode, const abt_vis_geometry* geo, int64_t nf_in, const int64_t* field_in,
                            double beam_mid_z, uint8_t* in_beam, uint8_t* is_vis, double* dist_beam,
                            int64_t* id_beam, uint8_t* is_shad)
{
    if (!geo) return abt_fail(ABT_ERR_ARG, "abt_find_vis: null geometry");
    if (mode != ABT_VIS_INT && mode != ABT_VIS_EXT && mode != ABT_VIS_INC)
        return abt_fail(ABT_ERR_ARG, "unknown visibility mode %d", mode);
    const int64_t nv = geo->nv, nf = geo->nf, na = geo->na;
    if (nv < 1 || nf < 1 || na < 1) return abt_fail(ABT_ERR_ARG, "abt_find_vis: need nv, nf, na >= 1");
    if (!geo->v || !geo->f_off || !geo->f_vi || !geo->f_mid || !geo->f_nz || !geo->f_ap || !geo->ap_nz ||
        !in_beam || !dist_beam || !id_beam || !is_shad)
        return abt_fail(ABT_ERR_ARG, "abt_find_vis: null array");
    if (nf >= (1LL << 31) / 3) return abt_fail(ABT_ERR_ARG, "abt_find_vis: too many facets (%lld)", (long long)nf);
    if (nv >= (1LL << 31)) return abt_fail(ABT_ERR_ARG, "abt_find_vis: too many vertices (%lld)", (long long)nv);
    if (geo->f_off[0] != 0) return abt_fail(ABT_ERR_ARG, "abt_find_vis: f_off[0] must be 0");
    for (int64_t i = 0; i < nf; i++) {
        if (geo->f_off[i + 1] - geo->f_off[i] < 3)
            return abt_fail(ABT_ERR_ARG, "abt_find_vis: facet %lld has fewer than 3 vertices", (long long)(i + 1));
        if (geo->f_ap[i] < 1 || geo->f_ap[i] > na)
            return abt_fail(ABT_ERR_ARG, "abt_find_vis: facet %lld aperture id %lld out of 1..%lld",
                            (long long)(i + 1), (long long)geo->f_ap[i], (long long)na);
    }
    const int64_t nvref = geo->f_off[nf];
    if (nvref >= (1LL << 31)) return abt_fail(ABT_ERR_ARG, "abt_find_vis: too many vertex references");
    for (int64_t k = 0; k < nvref; k++)
        if (geo->f_vi[k] < 1 || geo->f_vi[k] > nv)
            return abt_fail(ABT_ERR_ARG, "abt_find_vis: vertex id %lld out of 1..%lld", (long long)geo->f_vi[k],
                            (long long)nv);
    if (mode != ABT_VIS_INC) {
        if (nf_in < 1 || !field_in)
            return abt_fail(ABT_ERR_ARG, "abt_find_vis: the beam needs at least one illuminating facet");
        for (int64_t k = 0; k < nf_in; k++)
            if (field_in[k] < 1 || field_in[k] > nf)
                return abt_fail(ABT_ERR_ARG, "abt_find_vis: field_in facet %lld out of 1..%lld",
                                (long long)field_in[k], (long long)nf);
    } else {
        nf_in = 0;
    }
    // one staging buffer: inputs, outputs, workspace
    size_t o = 0;
    auto take = [&](size_t n) { const size_t at = o; o += up(n); return at; };
    const size_t o_v = take(sizeof(double) * 3 * nv), o_off = take(8 * (nf + 1)), o_vi = take(8 * nvref),
                 o_mid = take(sizeof(double) * 3 * nf), o_nz = take(8 * nf), o_ap = take(8 * nf),
                 o_apnz = take(8 * na), o_inoff = take(16), o_fin = take(8 * (nf_in > 0 ? nf_in : 1)),
                 o_bz = take(8), o_inb = take(nf), o_vis = take(nf), o_dist = take(8 * nf), o_id = take(8 * nf),
                 o_shad = take(nf);
    const size_t o_ws = o;
    o += layout(1, nf, nvref).total;
    hipStream_t st;
    void* p;
    int rc = abt_thread_staging(8, o, &st, &p);
    if (rc) return rc;
    char* d = (char*)p;
    // Inputs and results each in one copy through pinned memory (eleven and five small copies cost ~8 us each);
    // one by one where that cannot be had.
    char* pin = abt_thread_pinned(o_ws);
    const int64_t inoff[2] = {0, nf_in};
    const struct { size_t at; const void* from; size_t n; } in[] = {
        {o_v, geo->v, sizeof(double) * 3 * nv}, {o_off, geo->f_off, 8 * (size_t)(nf + 1)}, {o_vi, geo->f_vi, 8 * (size_t)nvref},
        {o_mid, geo->f_mid, sizeof(double) * 3 * nf}, {o_nz, geo->f_nz, 8 * (size_t)nf}, {o_ap, geo->f_ap, 8 * (size_t)nf},
        {o_apnz, geo->ap_nz, 8 * (size_t)na}, {o_inoff, inoff, 16}, {o_fin, field_in, 8 * (size_t)nf_in},
        {o_bz, &beam_mid_z, 8}};
    for (const auto& c : in) {
        if (!c.n) continue;
        if (pin) memcpy(pin + c.at, c.from, c.n);
        else HIPCHK(hipMemcpyAsync(d + c.at, c.from, c.n, hipMemcpyHostToDevice, st));
    }
    if (pin) HIPCHK(hipMemcpyAsync(d, pin, o_inb, hipMemcpyHostToDevice, st));
    abt_vis_batch a;
    a.mode = mode;
    a.nbeam = 1;
    a.nv = nv;
    a.nf = nf;
    a.na = na;
    a.f_off = (const int64_t*)(d + o_off);
    a.f_vi = (const int64_t*)(d + o_vi);
    a.f_ap = (const int64_t*)(d + o_ap);
    a.v = (const double*)(d + o_v);
    a.f_mid = (const double*)(d + o_mid);
    a.f_nz = (const double*)(d + o_nz);
    a.ap_nz = (const double*)(d + o_apnz);
    a.in_off = (const int64_t*)(d + o_inoff);
    a.field_in = (const int64_t*)(d + o_fin);
    a.beam_mid_z = (const double*)(d + o_bz);
    a.in_beam = (uint8_t*)(d + o_inb);
    a.is_vis = (uint8_t*)(d + o_vis);
    a.dist_beam = (double*)(d + o_dist);
    a.id_beam = (int64_t*)(d + o_id);
    a.is_shad = (uint8_t*)(d + o_shad);
    a.counts = nullptr;
    a.phases = 0;
    int cus = 0;
    rc = abt_ensure_device(&cus);
    if (!rc) rc = launch_all(a, nvref, d + o_ws, cus, st);
    if (rc) return rc;
    const struct { size_t at; void* to; size_t n; } out[] = {
        {o_inb, in_beam, (size_t)nf}, {o_vis, is_vis, (size_t)nf}, {o_dist, dist_beam, 8 * (size_t)nf},
        {o_id, id_beam, 8 * (size_t)nf}, {o_shad, is_shad, (size_t)nf}};
    if (pin) {
        HIPCHK(hipMemcpyAsync(pin + o_inb, d + o_inb, o_ws - o_inb, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        for (const auto& c : out)
            if (c.to) memcpy(c.to, pin + c.at, c.n);
        return 0;
    }
    for (const auto& c : out)
        if (c.to) HIPCHK(hipMemcpyAsync(c.to, d + c.at, c.n, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return 0;
}

// rotate()'s rotation for each beam (beam_loop_mod.f90:1488-1503), on the host with the C
// library's atan2, acos, sqrt and sincos like the reference (pi its REAL*4 literal,
// misc_submod.f90:12): R[9 b + 3 i + k] = rot(i+1, k+1).
extern "C" int abt_vis_rotations(int64_t nbeam, const double* prop, double* R)
{
#pragma clang fp contract(off)
    if (nbeam < 0 || (nbeam > 0 && (!prop || !R))) return abt_fail(ABT_ERR_ARG, "abt_vis_rotations: bad arguments");
    const double pi = 3.1415927410125732;
    for (int64_t b = 0; b < nbeam; b++) {
        const double* p = prop + 3 * b;
        double r1[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, r2[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, c, sn;
        const double th1 = 2 * pi - atan2(p[1], p[0]);
        sincos(th1, &sn, &c);
        r1[0] = c;
        r1[1] = -sn;
        r1[3] = sn;
        r1[4] = c;
        r1[8] = 1;
        double t[3];
        for (int i = 0; i < 3; i++) {
            double a = 0.0;
            for (int k = 0; k < 3; k++) a = a + r1[3 * i + k] * p[k];
            t[i] = a;
        }
        const double nrm = sqrt(t[0] * t[0] + t[1] * t[1] + t[2] * t[2]);   // normalise_vec (misc_submod.f90:2216-2227)
        for (int i = 0; i < 3; i++) t[i] = t[i] / nrm;
        sincos(acos(-t[2]), &sn, &c);
        r2[0] = c;
        r2[2] = sn;
        r2[6] = -sn;
        r2[8] = c;
        r2[4] = 1;
        for (int i = 0; i < 3; i++)
            for (int j = 0; j < 3; j++) {
                double a = 0.0;
                for (int k = 0; k < 3; k++) a = a + r2[3 * i + k] * r1[3 * k + j];
                R[9 * b + 3 * i + j] = a;
            }
    }
    return 0;
}

extern "C" int abt_vis_rotate_dev(int64_t nbeam, const double* rot, int64_t nv, const double* v0, int64_t nf,
                                  const double* mid0, const double* n0, int64_t na, const double* apn0, double* v,
                                  double* mid, double* nz, double* ap_nz, void* stream)
{
    using namespace abt::vis;
    if (nbeam < 0 || nv < 1 || nf < 1 || na < 1) return abt_fail(ABT_ERR_ARG, "abt_vis_rotate_dev: bad sizes");
    if (nbeam == 0) return 0;
    if (!rot || !v0 || !mid0 || !n0 || !apn0 || !v || !mid || !nz || !ap_nz)
        return abt_fail(ABT_ERR_ARG, "abt_vis_rotate_dev: null array");
    int rc = abt_ensure_device(nullptr);
    if (rc) return rc;
    const int64_t n = std::max(nv, std::max(nf, na));
    const unsigned gx = (unsigned)((n + BLK - 1) / BLK);
    for (int64_t b0 = 0; b0 < nbeam; b0 += BEAM_CHUNK) {
        const unsigned nb = (unsigned)std::min<int64_t>(BEAM_CHUNK, nbeam - b0);
        hipLaunchKernelGGL(k_vis_rotate, dim3(gx, nb), dim3(BLK), 0, (hipStream_t)stream, b0, rot, nv, v0, nf, mid0,
                           n0, na, apn0, v, mid, nz, ap_nz);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return abt_fail(ABT_ERR_HIP, "abt_vis_rotate_dev launch failed: %s", hipGetErrorString(e));
    return 0;
}
