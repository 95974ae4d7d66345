// adjoint.hip -- gradients of a loss of the orientation-averaged far field with
// respect to every aperture's vertices and amplitude matrix.
//
// Input: G = dL/dX_o per orientation and bin, X_o = k (ampl_far_beam + ampl_far_ext_diff)
// (the per-orientation total amplitude the batched forward writes).  Every beam b of
// orientation o (both trees) then has dL/dA_b = k G_o, and its gradients are sums over
// bins of per-(beam, bin) terms (adjbody.h).
//
// Work decomposition: one lane per beam, 64 lanes per unit, all lanes of a
// unit from one orientation and tree, so every lane reads the same bin at the same
// time: the bin's position and Lam' come through scalar loads and stay in scalar
// registers, the beam's constants and its 27 accumulators stay in vector registers, and
// no reduction across lanes is needed.  A unit may cover a chunk of the bins only (when
// there are too few beams to fill the chip); chunk partials are then summed in chunk
// order.  Every sum has a fixed order: results repeat bit for bit.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "adjbody.h"
#include "adjoint.h"

namespace abt {

constexpr int AL = 64;   // lanes of a unit (one wavefront)
constexpr int AW = 4;    // units of a workgroup of the FP64 kernel: they share the exponential table in LDS

// Lam' = k G T_phi^T per (orientation, bin), [o][bin][8]: FP64 in the eigenvectors of g I + h J
// (adj_lam_split), or FP32 plain for the mixed kernel; G in the batched forward's amplitude layout
// [o][8][nbins].
// T_phi = [[-s, -c], [c, -s]] (diff_mod.f90:646-650).
template <typename T>
__global__ __launch_bounds__(256) void k_adj_lam(const double* __restrict__ G, const double* __restrict__ cphi,
                                                 const double* __restrict__ sphi, int nphi, int nbins,
                                                 int norient, double k, T* __restrict__ lam)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)norient * nbins) return;
    const int o = (int)(i / nbins), bin = (int)(i - (int64_t)o * nbins);
    const int iphi = bin % nphi;
    const double c = cphi[iphi], s = sphi[iphi];
    const double* g = G + (int64_t)o * 8 * nbins + bin;
    double L[8];
#pragma unroll
    for (int q = 0; q < 8; q++) L[q] = k * g[(int64_t)q * nbins];
    T* out = lam + i * 8;
    double P[8];
    // pair (r, col): index 2 (r + 2 col)
#pragma unroll
    for (int r = 0; r < 2; r++)
#pragma unroll
        for (int ri = 0; ri < 2; ri++) {
            const double l1 = L[2 * r + ri], l2 = L[2 * (r + 2) + ri];
            P[2 * r + ri] = -s * l1 - c * l2;            // Lam'(r,1)
            P[2 * (r + 2) + ri] = c * l1 - s * l2;       // Lam'(r,2)
        }
    if (sizeof(T) == sizeof(double)) adj_lam_split(P, L);
#pragma unroll
    for (int q = 0; q < 8; q++) out[q] = sizeof(T) == sizeof(double) ? (T)L[q] : (T)P[q];
}

// Per-bin inputs, ADJ_BIN doubles.  Mixed: AdjBin; FP64: AdjFarBin's values, then the position at 8.
template <int PREC>
__global__ __launch_bounds__(256) void k_adj_bins(DevGrid g, double* __restrict__ bins)
{
    const int bin = blockIdx.x * 256 + threadIdx.x;
    if (bin >= g.nbins) return;
    const int bt = bin % g.nphi + g.nphi * g.theta_i;
    const AdjBin b{g.x[bin], g.y[bin], g.z[bin], g.x[bt], g.y[bt], g.rad[bin], g.kr_rev[bin]};
    double* o = bins + (int64_t)bin * ADJ_BIN;
    if (PREC == 0) {
        const AdjFarBin f = adj_far_bin(b);
        o[0] = f.f.nx; o[1] = f.f.ny; o[2] = f.f.nz; o[3] = f.f.ir;
        o[4] = f.xt; o[5] = f.yt; o[6] = f.kr;
        o[8] = b.x; o[9] = b.y; o[10] = b.z;
    } else {
        o[0] = b.x; o[1] = b.y; o[2] = b.z;
        o[3] = b.xt; o[4] = b.yt;
        o[5] = b.rad; o[6] = b.kr_rev;
    }
}

// Bins of a unit's chunk: never none, since the plan cuts nbins into at most nbins / 256 chunks and at most 64
__device__ __forceinline__ void chunk_bins(const AdjArgs& a, const AdjUnit& U, int* b0, int* b1)
{
    const int n = (a.nbins + a.nchunks - 1) / a.nchunks;
    *b0 = U.chunk * n;
    *b1 = min(a.nbins, *b0 + n);
}

// Per-beam gradients of one lane's sums to its row of the partials, [chunk][tree offset + beam][17].
__device__ __forceinline__ void store_beam(const AdjArgs& a, const AdjUnit& U, int64_t beam,
                                           const double* __restrict__ r, const AdjBeam& B, const AdjAcc& acc)
{
    double gv[9], ga[8];
    adj_finish(B, r + R_V20, r[R_SIGMA], acc, gv, ga);
    if (r[R_NV] != 3.0) {   // the adjoint covers triangular apertures only
#pragma unroll
        for (int q = 0; q < 9; q++) gv[q] = __builtin_nan("");
#pragma unroll
        for (int q = 0; q < 8; q++) ga[q] = __builtin_nan("");
    }
    const int64_t row = (U.tree ? a.nb_beam : 0) + beam;
    double* o = a.part + ((int64_t)U.chunk * a.nb_total + row) * 17;
#pragma unroll
    for (int q = 0; q < 9; q++) o[q] = gv[q];
#pragma unroll
    for (int q = 0; q < 8; q++) o[9 + q] = ga[q];
}

// Eight doubles through one scalar load: the bins' rows and Lam' are not written while the kernels run.  A lane's
// registers hold both kernels to two waves per SIMD, so the latency of a bin's inputs shows: their loads are
// issued a bin ahead (the mixed kernel's Lam' is not: its FP32 products would contract otherwise, and round so).
// 64 orientations of the rough column x 32,490 bins: FP64 168.4 -> 154.2 ms, mixed 149.7 -> 146.6.
typedef double Row8 __attribute__((ext_vector_type(8), aligned(8)));
__device__ __forceinline__ Row8 load_row(const double* p)
{
    return *(const __attribute__((address_space(4))) Row8*)(uintptr_t)p;
}

// FP64: AW units per workgroup, one per wave; two waves per SIMD, the beam's constants and sums
// in registers.
__global__ __launch_bounds__(AL * AW, 2) void k_adjoint64(AdjArgs a, int nunits)
{
    __shared__ double2 tab[ETAB_DOUBLES / 2];
    for (int i = threadIdx.x; i < ETAB_DOUBLES / 2; i += AL * AW)
        tab[i] = reinterpret_cast<const double2*>(a.etab)[i];
    __syncthreads();
    const int unit = blockIdx.x * AW + __builtin_amdgcn_readfirstlane(threadIdx.x / AL);
    if (unit >= nunits) return;
    const AdjUnit U = a.units[unit];
    const int lane = threadIdx.x % AL;
    const bool act = lane < U.count;
    const int64_t beam = U.start + (act ? lane : 0);
    const double* r = (U.tree ? a.recs_e : a.recs_b) + beam * REC;
    AdjBeam B;
    adj_beam_from_record(r, B);
    const bool far = B.cc <= a.cc_far;
    AdjSum sum;
    adj_zero_sum(sum);
    int b0, b1;
    chunk_bins(a, U, &b0, &b1);
    const double* lam = a.lam + (int64_t)U.o * a.nbins * 8;
    Row8 row = load_row(a.bins + (int64_t)b0 * ADJ_BIN), lrow = load_row(lam + (int64_t)b0 * 8);
    for (int i = b0; i < b1; i++) {
        const Row8 b = row, l = lrow;
        const int j = min(i + 1, b1 - 1);
        row = load_row(a.bins + (int64_t)j * ADJ_BIN);
        lrow = load_row(lam + (int64_t)j * 8);
        const AdjFarBin bn{{b[0], b[1], b[2], b[3]}, b[4], b[5], b[6], a.bins + (int64_t)i * ADJ_BIN + 8};
        const double lv[8] = {l[0], l[1], l[2], l[3], l[4], l[5], l[6], l[7]};
        adj_bin_far(B, bn, lv, far, reinterpret_cast<const double*>(tab), a.waveno, a.kt, sum);
    }
    if (!act) return;
    AdjAcc acc;
    adj_zero(acc);
    adj_add_sum(B, sum, acc);
    store_beam(a, U, beam, r, B, acc);
}

// Mixed: one unit per workgroup.
__global__ __launch_bounds__(AL, 2) void k_adjoint_mixed(AdjArgs a)
{
    const AdjUnit U = a.units[blockIdx.x];
    const int lane = threadIdx.x;
    const bool act = lane < U.count;
    const int64_t beam = U.start + (act ? lane : 0);
    const double* r = (U.tree ? a.recs_e : a.recs_b) + beam * REC;
    AdjBeam B;
    adj_beam_from_record(r, B);
    AdjAcc acc;
    adj_zero(acc);
    int b0, b1;
    chunk_bins(a, U, &b0, &b1);
    // FP32 partial sums over groups of ADJ_GROUP bins, added into FP64
    const float* lam = reinterpret_cast<const float*>(a.lam) + (int64_t)U.o * a.nbins * 8;
    Row8 row = load_row(a.bins + (int64_t)b0 * ADJ_BIN);
    for (int i0 = b0; i0 < b1; i0 += ADJ_GROUP) {
        AdjAccF af;
        adj_zero_f(af);
        const int i1 = min(b1, i0 + ADJ_GROUP);
        for (int i = i0; i < i1; i++) {
            const Row8 bb = row;
            const int j = min(i + 1, b1 - 1);
            row = load_row(a.bins + (int64_t)j * ADJ_BIN);
            const AdjBin bn{bb[0], bb[1], bb[2], bb[3], bb[4], bb[5], bb[6]};
            adj_bin_mixed(B, bn, lam + (int64_t)i * 8, a.waveno, a.lambda, af);
        }
        adj_add(acc, af);
    }
    if (act) store_beam(a, U, beam, r, B, acc);
}

// sum the chunk partials in chunk order and split them into the four outputs
__global__ __launch_bounds__(256) void k_adj_reduce(const double* __restrict__ part, int nchunks, int64_t nb_beam,
                                                    int64_t nb_total, double* gvb, double* gab, double* gve,
                                                    double* gae)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nb_total * 17) return;
    const int64_t row = i / 17;
    const int q = (int)(i - row * 17);
    double s = part[i];
    for (int c = 1; c < nchunks; c++) s += part[(int64_t)c * nb_total * 17 + i];
    const bool ext = row >= nb_beam;
    const int64_t b = ext ? row - nb_beam : row;
    if (q < 9) {
        double* o = ext ? gve : gvb;
        if (o) o[b * 9 + q] = s;
    } else {
        double* o = ext ? gae : gab;
        if (o) o[b * 8 + q - 9] = s;
    }
}

}  // namespace abt

using namespace abt;

extern "C" int abt_launch_adj_bins(const DevGrid* g, int prec, double* bins, hipStream_t st)
{
    const dim3 nb((unsigned)((g->nbins + 255) / 256));
    if (prec == 0)
        hipLaunchKernelGGL(k_adj_bins<0>, nb, dim3(256), 0, st, *g, bins);
    else
        hipLaunchKernelGGL(k_adj_bins<1>, nb, dim3(256), 0, st, *g, bins);
    return (int)hipGetLastError();
}

extern "C" int abt_launch_adjoint(const AdjArgs* a, int prec, int nunits, const double* G, const DevGrid* g,
                                  int norient, double* gvb, double* gab, double* gve, double* gae,
                                  hipStream_t st)
{
    const int64_t nl = (int64_t)norient * g->nbins;
    if (prec == 0)
        hipLaunchKernelGGL(k_adj_lam<double>, dim3((unsigned)((nl + 255) / 256)), dim3(256), 0, st, G, g->cphi,
                           g->sphi, g->nphi, g->nbins, norient, g->waveno, a->lam);
    else
        hipLaunchKernelGGL(k_adj_lam<float>, dim3((unsigned)((nl + 255) / 256)), dim3(256), 0, st, G, g->cphi,
                           g->sphi, g->nphi, g->nbins, norient, g->waveno, reinterpret_cast<float*>(a->lam));
    if (nunits > 0) {
        if (prec == 0)
            hipLaunchKernelGGL(k_adjoint64, dim3((nunits + AW - 1) / AW), dim3(AL * AW), 0, st, *a, nunits);
        else
            hipLaunchKernelGGL(k_adjoint_mixed, dim3(nunits), dim3(AL), 0, st, *a);
    }
    const int64_t n = a->nb_total * 17;
    if (n > 0)
        hipLaunchKernelGGL(k_adj_reduce, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                           (const double*)a->part, a->nchunks, a->nb_beam, a->nb_total, gvb, gab, gve, gae);
    return (int)hipGetLastError();
}
