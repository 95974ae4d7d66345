// far_field.hip -- coherent far-field sums of prepared beams onto the (theta, phi) bins.
//
// Work decomposition.  One lane per BPT far-field bins, bins contiguous with phi fastest (the
// Fortran (nphi, ntheta) layout), 256 lanes per workgroup.  A workgroup sums one segment of
// the beam list on one tile of 256 x BPT bins (grid: tiles x segments): every lane walks the
// beams in order, their records read through scalar loads.  Segment sums are stored as the body forms them; k_finish_sum
// (one orientation) or the batched plan's epilogue (batch.hip) adds them in segment order and
// finishes the sum, so each bin's sum is formed in a fixed order and repeats bit for bit.
// Cutting the beam list is what fills the chip when there are few bins or few orientations,
// and it bounds the last round of workgroups when there are many.  A single segment is finished
// in place.
//
// Bodies (ffbody.h, adjbody.h), by kernel precision:
//   0  the reference's formulas in FP64 (diffraction, diff_mod.f90:576-670; karczewski :124-198;
//      contour_integral :357-421), every phase formed with the reference's operations;
//   1  mixed: geometry, phases and their reduction in FP64, polarisation and the rotation-invariant
//      polygon form factor in FP32;
//   2  body 0 summing |amplitude|^2 instead (conditioning diagnostic);
//   3  the frame-free FP64 model (adjbody.h);
//   4  the mixed kernel's algorithm with every step in FP64.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include "sweep.h"

namespace abt {

constexpr int BLOCK = 256;

// A wave-uniform record through scalar loads: records are not written while a sweep runs, which the constant
// address space says (the loop's barriers would otherwise rule them out).
#if defined(__HIP_DEVICE_COMPILE__)
typedef const __attribute__((address_space(4))) double* ScalarRecord;
#else
typedef const double* ScalarRecord;
#endif
__device__ __forceinline__ ScalarRecord scalar_record(const double* r) { return (ScalarRecord)(uintptr_t)r; }

// A use of what the restructured body's geometry reads (centre, frame, direction, vertex count), so that it is
// loaded at once and waited for once: left to itself each piece is loaded where it is first used, three waits in a row
// before the phases.  24 orientations x 721 x 180 bins 86.8 -> 85.8 ms (on a slower card than ffbody.h's figures), 10,001 facets x 648,360 bins 30.85 ->
// 30.49.  With the vertices too 85.4, but 1 % slower where the field of view leaves most beams out; with the
// polarisation's values 86.6; in the mixed body 0.5 %: left as they are.  In the incoherent sum, whose lists are
// not cut and which waits for every record where bins are few, 5 % too: 4000 beams x 1332 bins 7.88 -> 7.13 ms.
__device__ __forceinline__ void geometry_together(ScalarRecord r)
{
    const ScalarRecord f = r + R_RR, c = r + R_COM;
    asm volatile("" : : "s"(c[0]), "s"(c[1]), "s"(c[2]), "s"(r[R_CC]), "s"(r[R_KT]), "s"(r[R_NV]), "s"(f[0]), "s"(f[1]),
                 "s"(f[2]), "s"(f[3]), "s"(f[4]), "s"(f[5]), "s"(f[6]), "s"(f[7]), "s"(f[8]), "s"(r[R_PROP2]),
                 "s"(r[R_PROP2 + 1]));
}

// Bin inputs of one lane slot.
template <int PREC>
__device__ __forceinline__ BinIn load_bin(const DevGrid& g, int bc)
{
    const int bt = bc % g.nphi + g.nphi * g.theta_i;   // the theta_i bin of the same phi
    BinIn bi;
    bi.x = g.x[bc]; bi.y = g.y[bc]; bi.z = g.z[bc];
    bi.xt = g.x[bt]; bi.yt = g.y[bt]; bi.zt = g.z[bt];
    bi.rad = PREC >= 3 ? g.rad[bc] : 0.0;
    return bi;
}

// Records.  A beam's record is the same for every lane, so it comes through scalar loads, straight into the
// FP64 (and FP32) instructions' scalar operands; TB beams at a time, a barrier apart, so that a workgroup's waves
// share the scalar cache's lines, and with the next TB records touched by one vector load a line, which
// brings them into L2 ahead of the scalar loads.  Each of the three counts: records from LDS kept it busy
// for 74 % of the time in the restructured body (42 % mixed, 51 % plain); scalar loads alone, or
// with the barriers alone, run the orientation averages at 109 and 108 ms (mixed 39 ms).  16 orientations x 361 x
// 180 bins, mixed: 30.8 -> 28.6 ms; 24 x 721 x 180, restructured: 98.5 -> 87.8 ms; 45 polygons x 721 x 180,
// plain: 190 -> 184 us a step.
// Occupancy: 4 waves per SIMD (128 VGPRs); 2 for two bins a lane and for the accurate body.  Two bins fit 3 (168 VGPRs),
// which the restructured body is told: with one register more it ran 32 orientations x 721 x 180 bins in 141 ms, not 115.
template <int PREC, int TB, int BPT, int MODE>
__global__ __launch_bounds__(BLOCK, BPT == 1 && PREC != 3 ? 4 : (PREC == 4 ? 3 : 2))
void k_sweep(SweepArgs a)
{
    constexpr bool INC = MODE == SWEEP_INC, LIST = MODE == SWEEP_LIST;
    // the exponential table, or the table with its low parts
    constexpr bool TAB = PREC == 0 || PREC == 2 || PREC == 4;
    __shared__ double etab[PREC == 4 ? ETAB_DOUBLES : (TAB ? ETAB_GRID : 1)];
    const DevGrid& g = a.g;
    const int tid = threadIdx.x;
    const int nslots = LIST ? *a.list_count : g.nbins;
    const int slot0 = blockIdx.x * (BLOCK * BPT) + tid;   // slot of lane j: slot0 + j * BLOCK
    if ((int)blockIdx.x * (BLOCK * BPT) >= nslots) return;   // LIST: tiles past the listed bins
    if (TAB) {   // published by the barriers of the beam loop before any use
        for (int q = tid; q < (PREC == 4 ? ETAB_DOUBLES : ETAB_GRID); q += BLOCK) etab[q] = g.etab[q];
    }
    BinIn bi[BPT];
    FarBin fb[BPT];
#pragma unroll
    for (int j = 0; j < BPT; j++) {
        const int sc = min(slot0 + j * BLOCK, nslots - 1);
        const int bc = LIST ? a.list[sc] : sc;
        bi[j] = load_bin<PREC>(g, bc);
        if (PREC == 4) fb[j] = far_bin(bi[j]);
    }
    double acc[BPT][8], inc[BPT];
#pragma unroll
    for (int j = 0; j < BPT; j++) {
        inc[j] = 0.0;
#pragma unroll
        for (int q = 0; q < 8; q++) acc[j][q] = 0.0;
    }
    const int seg = blockIdx.y;
    int64_t b0, b1;
    int tree = 0;
    if (a.segs) {
        const SweepSeg s = a.segs[seg];
        b0 = s.start;
        b1 = s.start + s.count;
        tree = s.tree;
    } else {
        b0 = (int64_t)seg * a.per;
        b1 = min(a.nb, b0 + a.per);
    }
    const double* __restrict__ recs = a.recs[tree];
    const double* __restrict__ vrecs = a.vrecs[tree];
    const auto touch = [&](int64_t t) {   // one lane per 128-byte line of the TB records from t
        const int64_t bytes = t < b1 ? min((int64_t)TB, b1 - t) * (REC * 8) : 0;
        int v = 0;
        if (tid * 128 < bytes) v = *reinterpret_cast<const int*>(reinterpret_cast<const char*>(recs + t * REC) + tid * 128);
        return v;
    };
    int line = touch(b0);
    for (int64_t t0 = b0; t0 < b1; t0 += TB) {
        const int nt = (int)min((int64_t)TB, b1 - t0);
        asm volatile("" : : "v"(line));   // a use: the load is kept, and has ended
        __syncthreads();
        line = touch(t0 + TB);
        if (PREC == 1) {
            // FP32 partial sums over groups of MIXED_GROUP beams (segments start at multiples of
            // it from the tree's first beam), added into FP64
            for (int g0 = 0; g0 < nt; g0 += MIXED_GROUP) {
                float accf[BPT][8], incf[BPT];
#pragma unroll
                for (int j = 0; j < BPT; j++) {
                    incf[j] = 0.f;
#pragma unroll
                    for (int q = 0; q < 8; q++) accf[j][q] = 0.f;
                }
                const int g1 = min(nt, g0 + MIXED_GROUP);
                for (int bb = g0; bb < g1; bb++) {
#pragma unroll
                    for (int j = 0; j < BPT; j++)
                        beam_bin_mixed_t<INC>(scalar_record(recs + (t0 + bb) * REC), vrecs, g, bi[j], a.fast_diff,
                                              accf[j], incf[j]);
                }
#pragma unroll
                for (int j = 0; j < BPT; j++) {
                    if (INC) inc[j] += (double)incf[j];
#pragma unroll
                    for (int q = 0; q < 8; q++) acc[j][q] += (double)accf[j][q];
                }
            }
        } else {
            for (int bb = 0; bb < nt; bb++) {
                if (PREC == 4 || PREC == 2) geometry_together(scalar_record(recs + (t0 + bb) * REC));
#pragma unroll
                for (int j = 0; j < BPT; j++) {
                    if (PREC == 4)
                        beam_bin_fp64r_far(scalar_record(recs + (t0 + bb) * REC), vrecs, fb[j], bi[j].xt, bi[j].yt, etab,
                                           g.cc_far, a.fast_diff, acc[j]);
                    else if (PREC == 3) {
                        AdjBeam B;
                        adj_beam_from_record(scalar_record(recs + (t0 + bb) * REC), B);
                        model_bin_fp64(B, bi[j].x, bi[j].y, bi[j].z, bi[j].xt, bi[j].yt, bi[j].rad, g.waveno,
                                       g.lambda, acc[j]);
                    } else
                        beam_bin_fp64p<PREC == 2>(scalar_record(recs + (t0 + bb) * REC), vrecs, g, bi[j], etab,
                                                  a.fast_diff, acc[j]);
                }
            }
        }
    }
    const int nbins = g.nbins;
#pragma unroll
    for (int j = 0; j < BPT; j++) {
        const int slot = slot0 + j * BLOCK;
        if (slot >= nslots) continue;
        if (a.part) {
            double* p = a.part + (int64_t)seg * 8 * nbins + slot;
#pragma unroll
            for (int q = 0; q < 8; q++) p[(int64_t)q * nbins] = acc[j][q];
            if (INC) a.ipart[(int64_t)seg * nbins + slot] = inc[j];
        } else if (PREC == 2) {   // incoherent intensity: one double per bin
            a.out[slot] = acc[j][0];
        } else {
            finish_sum<PREC>(acc[j], g, slot);
            double2* o2 = reinterpret_cast<double2*>(a.out);
#pragma unroll
            for (int q = 0; q < 4; q++) o2[slot + (int64_t)nbins * q] = make_double2(acc[j][2 * q], acc[j][2 * q + 1]);
        }
    }
}

// One orientation: the segment sums of a bin in segment order, finished, in the Fortran layout.
// Reads 64 bytes per bin and segment: bandwidth-bound.
template <int PREC>
__global__ __launch_bounds__(BLOCK) void k_finish_sum(DevGrid g, const double* __restrict__ part, int nseg,
                                                      double* __restrict__ out)
{
    const int bin = blockIdx.x * BLOCK + threadIdx.x;
    if (bin >= g.nbins) return;
    const int64_t nbins = g.nbins;
    double acc[8];
#pragma unroll
    for (int q = 0; q < 8; q++) acc[q] = 0.0;
#pragma unroll 4
    for (int s = 0; s < nseg; s++) {
        const double* p = part + (int64_t)s * 8 * nbins + bin;
#pragma unroll
        for (int q = 0; q < 8; q++) acc[q] += p[q * nbins];
    }
    finish_sum<PREC>(acc, g, bin);
    double2* o2 = reinterpret_cast<double2*>(out);
#pragma unroll
    for (int q = 0; q < 4; q++) o2[bin + nbins * q] = make_double2(acc[2 * q], acc[2 * q + 1]);
}

__global__ __launch_bounds__(BLOCK) void k_fill_zero(double* __restrict__ out, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i < n) out[i] = 0.0;
}

template <int PREC, int TB, int BPT, int MODE>
const void* sweep_kernel() { return reinterpret_cast<const void*>(&k_sweep<PREC, TB, BPT, MODE>); }

}  // namespace abt

// ---------------------------------------------------------------------------
// launch helpers (called by the runtime and the batched plan)

// Zero-fill of n doubles (a kernel, not hipMemsetAsync, so callers may capture it in a graph).
extern "C" int abt_launch_zero(double* out, int64_t n, hipStream_t st)
{
    if (n <= 0) return 0;
    hipLaunchKernelGGL(abt::k_fill_zero, dim3((unsigned)((n + abt::BLOCK - 1) / abt::BLOCK)),
                       dim3(abt::BLOCK), 0, st, out, n);
    return (int)hipGetLastError();
}

extern "C" const void* abt_sweep_kernel(int prec, int tb, int bpt, int mode)
{
    using namespace abt;
#define K(P, T, B, M) if (prec == P && tb == T && bpt == B && mode == M) return sweep_kernel<P, T, B, M>();
    K(0, 8, 1, 0) K(0, 16, 1, 0) K(0, 32, 1, 0) K(0, 8, 2, 0) K(0, 16, 2, 0) K(0, 32, 2, 0)
    K(1, 8, 1, 0) K(1, 16, 1, 0) K(1, 32, 1, 0) K(1, 8, 2, 0) K(1, 16, 2, 0) K(1, 32, 2, 0)
    K(1, 8, 1, 1) K(1, 16, 1, 1) K(1, 32, 1, 1) K(1, 8, 2, 1) K(1, 16, 2, 1) K(1, 32, 2, 1)
    K(2, 16, 1, 0)
    K(3, 16, 1, 0)
    K(4, 8, 1, 0) K(4, 16, 1, 0) K(4, 32, 1, 0) K(4, 8, 2, 0) K(4, 16, 2, 0)
    K(4, 16, 1, 2)
#undef K
    return nullptr;
}

extern "C" int abt_launch_sweep(const abt::SweepArgs* a, int nseg, int prec, int tb, int bpt, int mode,
                                hipStream_t st)
{
    const void* kern = abt_sweep_kernel(prec, tb, bpt, mode);
    if (!kern || nseg < 1 || nseg > 65535) return (int)hipErrorInvalidValue;
    abt::SweepArgs args = *a;
    void* params[] = {&args};
    const int64_t lanes = (int64_t)abt::BLOCK * bpt;
    const dim3 grid((unsigned)((a->g.nbins + lanes - 1) / lanes), (unsigned)nseg);
    return (int)hipLaunchKernel(kern, grid, dim3(abt::BLOCK), params, 0, st);
}

// One orientation's far field of nb prepared beams in nseg segments of `per` beams (a multiple
// of 8, so that the mixed body's FP32 beam groups do not depend on the cut); prec: the ABI's
// (0 plain FP64, 1 mixed, 3 restructured FP64) or 2, the incoherent sum (one segment).
// work: nseg * 64 bytes per bin when nseg > 1.
extern "C" int abt_launch_far_field(const abt::DevGrid* g, const double* recs, const double* vrecs,
                                    int64_t nb, int prec, int fast_diff, int64_t per, double* out, double* work,
                                    hipStream_t st)
{
    using namespace abt;
    if (g->nbins <= 0) return 0;
    const int kprec = prec == 3 ? 4 : prec;
    const int nseg = (int)((nb + per - 1) / per);
    SweepArgs a;
    memset(&a, 0, sizeof(a));
    a.g = *g;
    a.recs[0] = a.recs[1] = recs;
    a.vrecs[0] = a.vrecs[1] = vrecs;
    a.nb = nb;
    a.per = per;
    a.part = nseg > 1 ? work : nullptr;
    a.out = out;
    a.fast_diff = fast_diff;
    int e = abt_launch_sweep(&a, nseg, kprec, 16, 1, SWEEP_PLAIN, st);
    if (e) return e;
    if (nseg > 1) {
        const dim3 grid((g->nbins + BLOCK - 1) / BLOCK);
        const double* w = work;
        if (kprec == 0) hipLaunchKernelGGL(k_finish_sum<0>, grid, dim3(BLOCK), 0, st, *g, w, nseg, out);
        else if (kprec == 1) hipLaunchKernelGGL(k_finish_sum<1>, grid, dim3(BLOCK), 0, st, *g, w, nseg, out);
        else hipLaunchKernelGGL(k_finish_sum<4>, grid, dim3(BLOCK), 0, st, *g, w, nseg, out);
    }
    return (int)hipGetLastError();
}
