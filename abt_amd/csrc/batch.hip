// batch.hip -- orientation-averaged far field of many orientations.
//
// Replaces the orientation loop of the reference drivers (pbt_seq_mod.f90:146-269,
// pbt_mpi_mod.f90 over MPI ranks): per orientation diff_main (coherent sums of the
// beam tree and of the external-diffraction tree), finalise (amplitudes x k, total =
// beam + ext, Mueller matrices, phi/theta integrals; outputs_mod.f90:63-278) and
// summation (Mueller matrices summed incoherently over orientations,
// outputs_mod.f90:407-471).
//
// Work decomposition.  Every orientation's two beam lists are cut into segments of one length
// (the plan's, chosen so that segments x bin tiles are many workgroups per CU however few
// orientations or bins there are).  A run alternates, over groups of orientations whose segment
// sums fit the plan's buffer:
//   k_sweep (far_field.hip)  one workgroup per (segment, bin tile): the segment's coherent sum;
//   k_combine                one lane per bin: an orientation's segment sums added in beam order and
//                            finished, x k, the Mueller matrix of the total added to the chunk's
//                            sum, the bin's weighted S11 values added to the orientation's integrals.
// The segment sums cost 64 bytes per bin and segment written and read once, against ~10^3 beams of
// ~150 FP64 instructions in each: under 1 % of the time.  In return the sweep's loop has the
// registers and LDS to itself (an epilogue inside it held 73 spilled registers and 16 KB), and no
// shape leaves the chip idle.
// Against one persistent kernel that summed an orientation's whole beam list per bin tile (same body):
// 24 orientations x 721 x 180 bins 106.7 -> 100.2 ms, 16 x 361 x 180 in the mixed body 33.2 -> 28.0 ms,
// one orientation x 451 x 360 bins 12.3 -> 5.7 ms, 4 coarse orientations x 37 x 36 bins 1161 -> 103 us.
// Every output element is written by one lane, and every sum has a fixed order (beams, segments,
// orientations of a chunk, chunks, tiles), so results do not depend on scheduling and repeat bit
// for bit; the cut does not depend on the tile shape, so neither do the results.
//
// Per-orientation integrals (for the asymmetry parameters, which are ratios per
// orientation and so cannot be formed from the summed Mueller matrix):
//   I1 = sum_bins W1 S11,  I2 = sum_bins W2 S11,   for total, beam and ext,
// with W1 = wtheta(theta) sin(theta) wphi(phi) / k^2 and W2 = W1 cos(theta), where
// wtheta, wphi are the simpne weights of the theta and phi nodes: I1 is the
// orientation's scattering cross section (outputs_mod.f90:133-135) and I2 / I1 its
// asymmetry parameter (outputs_mod.f90:198-200).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "batch.h"
#include "mueller.h"

namespace abt {

constexpr int BB = 256;   // lanes per workgroup

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// The six integral terms of a workgroup's bins, summed in a fixed order into ip[0..5].
__device__ __forceinline__ void block_integrals(double v[6], double (*red)[6], double* __restrict__ ip)
{
    const int tid = threadIdx.x;
#pragma unroll
    for (int q = 0; q < 6; q++) v[q] = wave_sum(v[q]);
    __syncthreads();   // the previous orientation's sums have been read
    if ((tid & 63) == 0) {
#pragma unroll
        for (int q = 0; q < 6; q++) red[tid >> 6][q] = v[q];
    }
    __syncthreads();
    if (tid < 6) ip[tid] = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
}

__device__ __forceinline__ void integral_terms(const double xb[8], const double xe[8], double s11, double w1,
                                               double w2, double v[6])
{
    const double sb = mueller_s11(xb), se = mueller_s11(xe);
    v[0] = w1 * s11;
    v[1] = w2 * s11;
    v[2] = w1 * sb;
    v[3] = w2 * sb;
    v[4] = w1 * se;
    v[5] = w2 * se;
}

// The segment sums of one tree of one orientation added up in segment order, in place in the first
// (grid: components x bins, trees of the group).  Where trees have many segments there are few bins
// or few orientations, and k_combine's few lanes would walk them one load latency after another:
// 4 orientations x 27 segments x 1332 bins took 57 us in k_combine, 5 here and 9 there.
__global__ __launch_bounds__(BB) void k_sum_segments(double* __restrict__ part, double* __restrict__ inc,
                                                     const int32_t* __restrict__ seg_off, int sbase, int nbins)
{
    const int64_t n8 = (int64_t)8 * nbins;
    const int64_t i = (int64_t)blockIdx.x * BB + threadIdx.x;
    const int s0 = seg_off[blockIdx.y] - sbase, s1 = seg_off[blockIdx.y + 1] - sbase;
    if (s1 - s0 < 2 || i >= (inc ? n8 + nbins : n8)) return;
    const int64_t stride = i < n8 ? n8 : nbins;
    double* p = i < n8 ? part + s0 * n8 + i : inc + (int64_t)s0 * nbins + (i - n8);
    double s = p[0];
#pragma unroll 8
    for (int k = 1; k < s1 - s0; k++) s += p[k * stride];
    p[0] = s;
}

// Grid (ntiles of BB bins, nchunks): chunk c takes the c-th share of the group's orientations, in
// order, for one bin per lane.  Bandwidth-bound: 64 bytes per bin and segment read.
template <int PREC, int MODE>
__global__ __launch_bounds__(BB) void k_combine(CombineArgs a)
{
    constexpr bool INC = MODE == SWEEP_INC, LIST = MODE == SWEEP_LIST;
    __shared__ double red[BB / 64][6];
    const int nbins = a.g.nbins;
    const int nslots = LIST ? *a.list_count : nbins;
    const int t = blockIdx.x, c = blockIdx.y;
    if (t * BB >= nslots) return;   // uniform over the workgroup
    const int slot = t * BB + threadIdx.x;
    const bool live = slot < nslots;
    const int sc = live ? slot : nslots - 1;
    const int bc = LIST ? a.list[sc] : sc;
    const double k = a.g.waveno;
    const double w1 = LIST ? 0.0 : a.w1[bc], w2 = LIST ? 0.0 : a.w2[bc];
    double msum[16], esum = 0.0;
#pragma unroll
    for (int e = 0; e < 16; e++) msum[e] = 0.0;
    const int n = a.o1 - a.o0;
    const int oa = a.o0 + (int)((int64_t)n * c / a.nchunks), ob = a.o0 + (int)((int64_t)n * (c + 1) / a.nchunks);
    const int sbase = a.seg_off[2 * a.o0];   // the buffer holds the group's segments from its first
    for (int o = oa; o < ob; o++) {
        double xb[8], xe[8], xt[8], m[16], inc = 0.0;
#pragma unroll
        for (int tree = 0; tree < 2; tree++) {
            double acc[8];
#pragma unroll
            for (int q = 0; q < 8; q++) acc[q] = 0.0;
            const int s0 = a.seg_off[2 * o + tree] - sbase;
            const int s1 = a.summed ? min(s0 + 1, a.seg_off[2 * o + tree + 1] - sbase)
                                    : a.seg_off[2 * o + tree + 1] - sbase;
            for (int s = s0; s < s1; s++) {
                const double* p = a.part + (int64_t)s * 8 * nbins + sc;
#pragma unroll
                for (int q = 0; q < 8; q++) acc[q] += p[(int64_t)q * nbins];
                if (INC) inc += a.ipart_inc[(int64_t)s * nbins + sc];
            }
            finish_sum<PREC>(acc, a.g, bc);
#pragma unroll
            for (int q = 0; q < 8; q++) (tree ? xe : xb)[q] = acc[q] * k;   // outputs_mod.f90:104-105
        }
#pragma unroll
        for (int q = 0; q < 8; q++) xt[q] = xb[q] + xe[q];                  // outputs_mod.f90:108
        mueller16(xt, m);
#pragma unroll
        for (int e = 0; e < 16; e++) msum[e] += m[e];
        if (INC) esum += m[0] * (inc * (k * k));
        if (live && a.store) {
            double* so = a.store + (int64_t)o * 16 * nbins + bc;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                so[(int64_t)q * nbins] = xb[q];
                so[(int64_t)(8 + q) * nbins] = xe[q];
            }
        }
        if (live && a.ampl_out) {
            double* ao = a.ampl_out + (int64_t)o * 8 * nbins + bc;
#pragma unroll
            for (int q = 0; q < 8; q++) ao[(int64_t)q * nbins] = xt[q];
        }
        if (!LIST) {
            double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            if (live) integral_terms(xb, xe, m[0], w1, w2, v);
            block_integrals(v, red, a.ipart + ((int64_t)o * gridDim.x + t) * 6);
        }
    }
    if (!live) return;
    if (a.mpart) {
        double* mo = a.mpart + (int64_t)c * 16 * nbins + slot;
#pragma unroll
        for (int e = 0; e < 16; e++) mo[(int64_t)e * nbins] = a.first ? msum[e] : mo[(int64_t)e * nbins] + msum[e];
    }
    if (INC) {
        double* ep = a.epart + (int64_t)c * nbins + slot;
        *ep = a.first ? esum : *ep + esum;
    }
}

// mueller[e][bin] = sum over chunks, in chunk order
__global__ __launch_bounds__(BB) void k_batch_reduce_m(const double* __restrict__ mpart, int nchunks,
                                                       int64_t n, double* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * BB + threadIdx.x;
    if (i >= n) return;
    double s = mpart[i];
    for (int c = 1; c < nchunks; c++) s += mpart[(int64_t)c * n + i];
    out[i] = s;
}

// integrals[o][q] = sum over tiles: one wave per (orientation, integral), each lane every 64th tile
// in order, then the lanes (a serial walk over the 507 tiles of a 721 x 180 grid took 79 us)
__global__ __launch_bounds__(BB) void k_batch_reduce_i(const double* __restrict__ ipart, int ntiles,
                                                       int norient, double* __restrict__ out)
{
    const int i = blockIdx.x * (BB / 64) + (threadIdx.x >> 6);
    if (i >= norient * 6) return;
    const int o = i / 6, q = i - 6 * o;
    const double* p = ipart + (int64_t)o * ntiles * 6 + q;
    double s = 0.0;
    for (int t = threadIdx.x & 63; t < ntiles; t += 64) s += p[(int64_t)t * 6];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) out[i] = s;
}

// mueller_1d(theta, e) = the phi integral (get_1d_mueller, outputs_mod.f90:280-329) of the summed
// Mueller matrix; the reference sums the per-orientation 1-D matrices, which is the same linear map
// applied before the sum.  One wave per (element, theta): the row's values times the nodes' weights.
__global__ __launch_bounds__(BB) void k_batch_phi(const double* __restrict__ M, const double* __restrict__ wphi,
                                                  int nphi, int ntheta, double* __restrict__ out)
{
    const int row = blockIdx.x * (BB / 64) + (threadIdx.x >> 6);
    if (row >= 16 * ntheta) return;
    const double* y = M + (int64_t)row * nphi;
    double s = 0.0;
    for (int i = threadIdx.x & 63; i < nphi; i += 64) s = fma(wphi[i], y[i], s);
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) out[row] = s;
}

// ---- -scaling (outputs_mod.f90:146-184) ----------------------------------------
//
// Per orientation the reference divides the beam amplitudes by sqrt(scatt_beam /
// beam_energy_out) and the ext amplitudes by sqrt(scatt_ext_diff / ext_energy_out), scatt_*
// being that orientation's own cross sections, then remakes the Mueller matrices and the
// integrated parameters.  The cross sections need every bin of the orientation, so the
// first pass stores the amplitudes, and this pass divides and sums them.

// div[o] = {sqrt(scatt_beam / E_beam), sqrt(scatt_ext / E_ext)} from the unscaled integrals
__global__ __launch_bounds__(BB) void k_scale_div(const double* __restrict__ raw, const double* __restrict__ eb,
                                                  const double* __restrict__ ee, int norient,
                                                  double* __restrict__ div)
{
    const int o = blockIdx.x * BB + threadIdx.x;
    if (o >= norient) return;
    div[2 * o] = sqrt(raw[6 * o + 2] / eb[o]);
    div[2 * o + 1] = sqrt(raw[6 * o + 4] / ee[o]);
}

// grid (ntiles of BB bins, nchunks): chunk c's share of the orientations in order for one bin per
// lane; the Mueller sum into mpart[c] and the integrals into ipart[o][t], as k_combine writes them.
__global__ __launch_bounds__(BB) void k_batch_scaled(CombineArgs a, const double* __restrict__ div)
{
    __shared__ double red[BB / 64][6];
    const int tid = threadIdx.x;
    const int nbins = a.g.nbins;
    const int t = blockIdx.x, c = blockIdx.y;
    const int bc = t * BB + tid;
    const bool live = bc < nbins;
    const int b = live ? bc : nbins - 1;
    const double w1 = a.w1[b], w2 = a.w2[b];
    double msum[16];
#pragma unroll
    for (int e = 0; e < 16; e++) msum[e] = 0.0;
    const int o0 = (int)((int64_t)a.o1 * c / a.nchunks), o1 = (int)((int64_t)a.o1 * (c + 1) / a.nchunks);
    for (int o = o0; o < o1; o++) {
        const double db = div[2 * o], de = div[2 * o + 1];
        const double* so = a.store + (int64_t)o * 16 * nbins + b;
        double xb[8], xe[8], xt[8], m[16];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            xb[q] = so[(int64_t)q * nbins] / db;          // outputs_mod.f90:151
            xe[q] = so[(int64_t)(8 + q) * nbins] / de;    // outputs_mod.f90:154
            xt[q] = xb[q] + xe[q];                        // outputs_mod.f90:156
        }
        mueller16(xt, m);
#pragma unroll
        for (int e = 0; e < 16; e++) msum[e] += m[e];
        if (live && a.ampl_out) {
            double* ao = a.ampl_out + (int64_t)o * 8 * nbins + bc;
#pragma unroll
            for (int q = 0; q < 8; q++) ao[(int64_t)q * nbins] = xt[q];
        }
        double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if (live) integral_terms(xb, xe, m[0], w1, w2, v);
        block_integrals(v, red, a.ipart + ((int64_t)o * gridDim.x + t) * 6);
    }
    if (live) {
        double* mo = a.mpart + (int64_t)c * 16 * nbins + bc;
#pragma unroll
        for (int e = 0; e < 16; e++) mo[(int64_t)e * nbins] = msum[e];
    }
}

// ---- gated mixed precision ---------------------------------------------------
//
// The FP32 body's rounding makes each orientation's amplitude carry a relative error of
// ~1e-7 of the bin's incoherent beam sum; summed over orientations with independent
// signs, the error of a Mueller element of the orientation sum is bounded by
// EST_C * sqrt(sum_o S11_o I_o) (calibrated on the rough-column and absorbing-column
// workloads against the FP64 reference, with a margin).  A bin is recomputed in FP64 when
// that bound exceeds the accuracy gate of one of its elements:
//   |dS_11| <= GATE_S11 S11,   |dS_ij| <= GATE_ELEM max(|S_ij|, GATE_FLOOR S11).
constexpr double EST_C = 5.0e-7;
constexpr double GATE_S11 = 1.0e-6;
constexpr double GATE_ELEM = 1.0e-5;
constexpr double GATE_FLOOR = 1.0e-3;

__global__ __launch_bounds__(BB) void k_gate_flags(const double* __restrict__ M, const double* __restrict__ est,
                                                   int nbins, int32_t* __restrict__ flags)
{
    const int b = blockIdx.x * BB + threadIdx.x;
    if (b >= nbins) return;
    const double s11 = fabs(M[b]);
    double mn = s11;
    for (int e = 1; e < 16; e++) mn = fmin(mn, fabs(M[(int64_t)e * nbins + b]));
    const double bound = EST_C * sqrt(fmax(est[b], 0.0));
    const double tol = fmin(GATE_S11 * s11, GATE_ELEM * fmax(mn, GATE_FLOOR * s11));
    // NaN anywhere (bound or tolerance) also sends the bin to FP64
    flags[b] = !(bound <= tol);
}

// Flagged bins in ascending order: one workgroup, each lane a contiguous segment.
constexpr int CB = 1024;
__global__ __launch_bounds__(CB) void k_gate_compact(const int32_t* __restrict__ flags, int nbins,
                                                     int32_t* __restrict__ list, int32_t* __restrict__ count)
{
    __shared__ int32_t sc[CB];
    const int tid = threadIdx.x;
    const int per = (nbins + CB - 1) / CB;
    const int b0 = min(nbins, tid * per), b1 = min(nbins, b0 + per);
    int n = 0;
    for (int b = b0; b < b1; b++) n += flags[b];
    sc[tid] = n;
    __syncthreads();
    for (int off = 1; off < CB; off <<= 1) {   // inclusive scan
        const int v = tid >= off ? sc[tid - off] : 0;
        __syncthreads();
        sc[tid] += v;
        __syncthreads();
    }
    int pos = sc[tid] - n;
    for (int b = b0; b < b1; b++)
        if (flags[b]) list[pos++] = b;
    if (tid == CB - 1) *count = sc[CB - 1];
}

// mueller[e][list[i]] = sum over chunks of the list pass's partials (chunk order)
__global__ __launch_bounds__(BB) void k_gate_scatter(const double* __restrict__ mpart, int nchunks, int nbins,
                                                     const int32_t* __restrict__ list,
                                                     const int32_t* __restrict__ count, double* __restrict__ out)
{
    const int64_t idx = (int64_t)blockIdx.x * BB + threadIdx.x;   // over 16 * nbins
    const int e = (int)(idx / nbins);
    const int i = (int)(idx - (int64_t)e * nbins);
    if (e >= 16 || i >= *count) return;
    const int64_t stride = (int64_t)16 * nbins;
    const double* p = mpart + (int64_t)e * nbins + i;
    double s = p[0];
    for (int c = 1; c < nchunks; c++) s += p[c * stride];
    out[(int64_t)e * nbins + list[i]] = s;
}

}  // namespace abt

// ---------------------------------------------------------------------------
// launch sequences (called by the plan): kernels only, so callers may capture them in a graph
namespace {

using namespace abt;

unsigned blocks(int64_t n) { return (unsigned)((n + BB - 1) / BB); }

template <int MODE>
void launch_combine(int prec, const CombineArgs& a, hipStream_t st)
{
    const dim3 grid(blocks(a.g.nbins), (unsigned)a.nchunks);
    if (MODE == SWEEP_INC) hipLaunchKernelGGL((k_combine<1, SWEEP_INC>), grid, dim3(BB), 0, st, a);
    else if (MODE == SWEEP_LIST) hipLaunchKernelGGL((k_combine<4, SWEEP_LIST>), grid, dim3(BB), 0, st, a);
    else if (prec == 0) hipLaunchKernelGGL((k_combine<0, SWEEP_PLAIN>), grid, dim3(BB), 0, st, a);
    else if (prec == 1) hipLaunchKernelGGL((k_combine<1, SWEEP_PLAIN>), grid, dim3(BB), 0, st, a);
    else if (prec == 3) hipLaunchKernelGGL((k_combine<3, SWEEP_PLAIN>), grid, dim3(BB), 0, st, a);
    else hipLaunchKernelGGL((k_combine<4, SWEEP_PLAIN>), grid, dim3(BB), 0, st, a);
}

// Sweep and epilogue of every group of the run's orientations.
template <int MODE>
int run_groups(const BatchRun& r, int prec, int tb, int bpt, SweepArgs sw, CombineArgs cb)
{
    for (int i = 0; i < r.ngroups; i++) {
        const BatchGroup& G = r.groups[i];
        if (G.s1 > G.s0) {   // a group may have no beams at all
            SweepArgs s = sw;
            s.segs = r.sweep.segs + G.s0;
            int e = abt_launch_sweep(&s, G.s1 - G.s0, prec, tb, bpt, MODE, r.st);
            if (e) return e;
        }
        // trees of many segments: summed by their own kernel first
        const bool sum = (G.s1 - G.s0) > 4 * (G.o1 - G.o0);
        if (sum) {
            const int64_t n = (int64_t)(MODE == SWEEP_INC ? 9 : 8) * cb.g.nbins;
            hipLaunchKernelGGL(k_sum_segments, dim3(blocks(n), (unsigned)(2 * (G.o1 - G.o0))), dim3(BB), 0, r.st,
                               sw.part, MODE == SWEEP_INC ? sw.ipart : (double*)nullptr, cb.seg_off + 2 * G.o0, G.s0,
                               cb.g.nbins);
        }
        CombineArgs c = cb;
        c.summed = sum;
        c.o0 = G.o0;
        c.o1 = G.o1;
        c.nchunks = r.nchunks;
        c.first = i == 0;
        launch_combine<MODE>(prec, c, r.st);
    }
    return (int)hipGetLastError();
}

void reduce_mueller(const BatchRun& r)
{
    const int64_t n = (int64_t)16 * r.comb.g.nbins;
    if (r.nchunks > 1)
        hipLaunchKernelGGL(k_batch_reduce_m, dim3(blocks(n)), dim3(BB), 0, r.st, (const double*)r.mpart, r.nchunks, n,
                           r.mueller);
}

void reduce_integrals(const BatchRun& r, double* out)
{
    hipLaunchKernelGGL(k_batch_reduce_i, dim3((unsigned)((r.norient * 6 + 3) / 4)), dim3(BB), 0, r.st,
                       (const double*)r.comb.ipart, (int)blocks(r.comb.g.nbins), r.norient, out);
}

void phi_integral(const BatchRun& r)
{
    const DevGrid& g = r.comb.g;
    if (r.mueller_1d)
        hipLaunchKernelGGL(k_batch_phi, dim3((unsigned)((16 * g.ntheta + BB / 64 - 1) / (BB / 64))), dim3(BB), 0, r.st,
                           (const double*)r.mueller, r.wphi, g.nphi, g.ntheta, r.mueller_1d);
}

CombineArgs with_mueller(const BatchRun& r)
{
    CombineArgs c = r.comb;
    c.mpart = r.nchunks > 1 ? r.mpart : r.mueller;
    return c;
}

}  // namespace

extern "C" int abt_launch_batch(const BatchRun* r)
{
    int e = run_groups<SWEEP_PLAIN>(*r, r->prec, r->tb, r->bpt, r->sweep, with_mueller(*r));
    if (e) return e;
    reduce_mueller(*r);
    reduce_integrals(*r, r->integrals);
    phi_integral(*r);
    return (int)hipGetLastError();
}

extern "C" int abt_launch_batch_scaled(const BatchRun* r, const ScaleBufs* s)
{
    if (!s->store) return (int)hipErrorInvalidValue;
    CombineArgs c = r->comb;
    c.mpart = nullptr;      // formed from the divided amplitudes below
    c.ampl_out = nullptr;
    c.store = s->store;
    int e = run_groups<SWEEP_PLAIN>(*r, r->prec, r->tb, r->bpt, r->sweep, c);
    if (e) return e;
    reduce_integrals(*r, s->raw);
    hipLaunchKernelGGL(k_scale_div, dim3(blocks(r->norient)), dim3(BB), 0, r->st, (const double*)s->raw,
                       s->beam_energy, s->ext_energy, r->norient, s->div);
    c = with_mueller(*r);
    c.store = s->store;
    c.o0 = 0;
    c.o1 = r->norient;
    c.nchunks = r->nchunks;
    hipLaunchKernelGGL(k_batch_scaled, dim3(blocks(c.g.nbins), (unsigned)r->nchunks), dim3(BB), 0, r->st, c,
                       (const double*)s->div);
    reduce_mueller(*r);
    reduce_integrals(*r, r->integrals);
    phi_integral(*r);
    return (int)hipGetLastError();
}

extern "C" int abt_launch_batch_est(const BatchRun* r, const GateBufs* q)
{
    CombineArgs c = with_mueller(*r);
    c.epart = r->nchunks > 1 ? q->epart : q->est;
    return run_groups<SWEEP_INC>(*r, 1, r->tb, r->bpt, r->sweep, c);
}

extern "C" int abt_launch_batch_gated(const BatchRun* r, const GateBufs* q)
{
    // pass 1: mixed, with the error scale
    int e = abt_launch_batch_est(r, q);
    if (e) return e;
    const int nbins = r->comb.g.nbins;
    reduce_mueller(*r);
    if (r->nchunks > 1)
        hipLaunchKernelGGL(k_batch_reduce_m, dim3(blocks(nbins)), dim3(BB), 0, r->st, (const double*)q->epart,
                           r->nchunks, (int64_t)nbins, q->est);
    reduce_integrals(*r, r->integrals);
    // the bins whose error bound exceeds the gate
    hipLaunchKernelGGL(k_gate_flags, dim3(blocks(nbins)), dim3(BB), 0, r->st, (const double*)r->mueller,
                       (const double*)q->est, nbins, q->flags);
    hipLaunchKernelGGL(k_gate_compact, dim3(1), dim3(CB), 0, r->st, (const int32_t*)q->flags, nbins, q->list, q->count);
    // pass 2: those bins in FP64 (restructured body), written over the mixed sums
    SweepArgs s = r->sweep;
    s.list = q->list;
    s.list_count = q->count;
    CombineArgs c = r->comb;
    c.mpart = q->lpart;
    c.list = q->list;
    c.list_count = q->count;
    e = run_groups<SWEEP_LIST>(*r, 4, 16, 1, s, c);
    if (e) return e;
    hipLaunchKernelGGL(k_gate_scatter, dim3(blocks((int64_t)16 * nbins)), dim3(BB), 0, r->st, (const double*)q->lpart,
                       r->nchunks, nbins, (const int32_t*)q->list, (const int32_t*)q->count, r->mueller);
    phi_integral(*r);
    return (int)hipGetLastError();
}
