// mueller.hip -- far-field epilogue of one orientation on the device:
// finalise (outputs_mod.f90:63-278): amplitudes x k, total = beam + ext,
// ampl_to_mueller for total/beam/ext (outputs_mod.f90:473-549, Bohren & Huffman
// 3.16), phi integration by simpne (get_1d_mueller, outputs_mod.f90:280-329;
// simpne misc_submod.f90:2392-2531), theta integrals (scattering cross
// sections, asymmetry parameters, back-scattering) and the optional energy
// scaling (outputs_mod.f90:146-184).  FP64 throughout; amplitudes and matrices
// with contraction off, so that they round like the reference, the integrals as
// weighted sums in a fixed order.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "../../include/abt_diff.h"
#include "mueller.h"
#include "records.h"
#include "rt_internal.h"
#include "simpne.h"

namespace abt {

constexpr int MB = 256;

// a complex amplitude; a caller's array need not be aligned beyond its doubles
typedef double Pair __attribute__((ext_vector_type(2), aligned(8)));

// One bin's amplitudes: k ampl, divided by the energy scaling factor where there is one (the
// reference's two steps).
__device__ __forceinline__ void load_ampl(const Pair* __restrict__ A, int64_t b, int64_t nb, double k,
                                          const double* __restrict__ f, double s[8])
{
#pragma clang fp contract(off)
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const Pair v = A[b + nb * q];
        s[2 * q] = v.x * k;
        s[2 * q + 1] = v.y * k;
    }
    if (f) {
        const double d = *f;
#pragma unroll
        for (int q = 0; q < 8; q++) s[q] = s[q] / d;
    }
}

__device__ __forceinline__ void store_ampl(Pair* __restrict__ A, int64_t b, int64_t nb, const double s[8])
{
#pragma unroll
    for (int q = 0; q < 4; q++) A[b + nb * q] = Pair{s[2 * q], s[2 * q + 1]};
}

// Adds N values over a wave by halving: lanes a bit apart keep one half of the values each and pass the
// other, so 48 values take 24 + 12 + 6 + 3 exchanges and two rounds of 3 instead of six rounds of
// 48.  v[0 .. N/16) holds the sums of the values at N/2 b0 + N/4 b1 + N/8 b2 + N/16 b3, b the lane's bits.
template <int N, int BIT>
__device__ __forceinline__ void wave_sums(double* v, int lane)
{
    if constexpr (BIT < 4) {
        const bool up = (lane >> BIT) & 1;
#pragma unroll
        for (int i = 0; i < N / 2; i++) {
            const double keep = up ? v[i + N / 2] : v[i], give = up ? v[i] : v[i + N / 2];
            v[i] = keep + __shfl_xor(give, 1 << BIT);
        }
        wave_sums<N / 2, BIT + 1>(v, lane);
    } else if constexpr (BIT < 6) {
#pragma unroll
        for (int i = 0; i < N; i++) v[i] += __shfl_xor(v[i], 1 << BIT);
        wave_sums<N, BIT + 1>(v, lane);
    }
}

// The epilogue of one theta per workgroup, a lane per phi: the scaled amplitudes, the three Mueller
// matrices (total, beam, ext) and their phi integrals (simpne as weights) in one pass over the bins.
// Bound by its writes, 512 of 640 bytes a bin.  FULL = false: the phi integrals of S11 of beam and
// ext alone, for the energy scaling factors; nothing else is written.
// 721 theta x 180 phi with energy scaling, all kernels of the epilogue: 420 -> 31 us.  Before, eight kernels:
// amplitudes, matrices and integrals apart (the integrals a lane per theta and element, uncoalesced,
// 34 us a pass), and the theta integrals as three serial chains of 721 (146 us a pass).
template <bool FULL>
__global__ __launch_bounds__(MB) void k_epilogue(DevGrid g, double* __restrict__ ab, double* __restrict__ ae,
                                                 const double* __restrict__ f, double* __restrict__ M,
                                                 double* __restrict__ m1d)
{
#pragma clang fp contract(off)
    constexpr int NS = FULL ? 48 : 16;   // sums (FULL = false: 2 used)
    __shared__ double part[MB / 64][NS];
    const int64_t nb = g.nbins;
    const int nph = g.nphi, nth = g.ntheta, j = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    Pair* B = reinterpret_cast<Pair*>(ab);
    Pair* E = reinterpret_cast<Pair*>(ae);
    double acc[NS];
#pragma unroll
    for (int e = 0; e < NS; e++) acc[e] = 0.0;
    for (int i = threadIdx.x; i < nph; i += blockDim.x) {
        const int64_t b = (int64_t)nph * j + i;
        const double w = g.wphi[i];
        double sb[8], se[8];
        load_ampl(B, b, nb, g.waveno, f, sb);
        load_ampl(E, b, nb, g.waveno, f ? f + 1 : f, se);
        if (FULL) {
            store_ampl(B, b, nb, sb);
            store_ampl(E, b, nb, se);
            double st[8];
#pragma unroll
            for (int q = 0; q < 8; q++) st[q] = sb[q] + se[q];
#pragma unroll
            for (int m = 0; m < 3; m++) {
                double mm[16];
                mueller16(m == 0 ? st : (m == 1 ? sb : se), mm);
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    M[b + nb * (16 * m + e)] = mm[e];
                    acc[16 * m + e] += w * mm[e];
                }
            }
        } else {
            acc[0] += w * mueller_s11(sb);
            acc[1] += w * mueller_s11(se);
        }
    }
    if (FULL) {
        wave_sums<NS, 0>(acc, lane);
        if (lane < 16) {
            const int o = 24 * (lane & 1) + 12 * ((lane >> 1) & 1) + 6 * ((lane >> 2) & 1) + 3 * (lane >> 3);
#pragma unroll
            for (int e = 0; e < NS / 16; e++) part[wave][o + e] = acc[e];
        }
    } else {
        wave_sums<2, 4>(acc, lane);
#pragma unroll
        for (int o = 1; o < 16; o *= 2) {
            acc[0] += __shfl_xor(acc[0], o);
            acc[1] += __shfl_xor(acc[1], o);
        }
        if (lane == 0) {
            part[wave][0] = acc[0];
            part[wave][1] = acc[1];
        }
    }
    __syncthreads();
    const int nw = blockDim.x >> 6;
    if (threadIdx.x < (FULL ? 48 : 2)) {
        double s = part[0][threadIdx.x];
        for (int q = 1; q < nw; q++) s += part[q][threadIdx.x];
        // [matrix][element][theta]; FULL = false: S11 of beam and ext
        const int row = FULL ? threadIdx.x : 16 * (threadIdx.x + 1);
        m1d[(int64_t)nth * row + j] = s;
    }
}

// Theta integrals (outputs_mod.f90:133-135, 198-205) from the phi integrals of S11, as weighted sums over one
// workgroup: scattering cross sections and asymmetry parameters; back-scattering.
// params: scatt, scatt_beam, scatt_ext, g, g_beam, g_ext, back_scatt, f_beam, f_ext.
// FACTORS: the energy scaling factors sqrt(scatt_x / energy_x) into params[7..8] alone.
template <bool FACTORS>
__global__ __launch_bounds__(MB) void k_theta_params(DevGrid g, const double* __restrict__ m1d,
                                                     const double* __restrict__ M, double ebeam, double eext,
                                                     double* __restrict__ params)
{
    __shared__ double part[MB / 64][6];
    const int tid = threadIdx.x, nth = g.ntheta;
    double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int j = tid; j < nth; j += MB) {
        const double w = g.wth[j], wc = g.wth[nth + j];
#pragma unroll
        for (int m = FACTORS ? 1 : 0; m < 3; m++) {
            const double v = m1d[(int64_t)16 * nth * m + j];
            s[m] += w * v;
            if (!FACTORS) s[3 + m] += wc * v;
        }
    }
#pragma unroll
    for (int q = 0; q < 6; q++) {
#pragma unroll
        for (int o = 1; o < 64; o *= 2) s[q] += __shfl_xor(s[q], o);
        if ((tid & 63) == 0) part[tid >> 6][q] = s[q];
    }
    __syncthreads();
    if (tid >= 3) return;
    double sc = 0.0, gc = 0.0;
    for (int q = 0; q < MB / 64; q++) {
        sc += part[q][tid];
        gc += part[q][3 + tid];
    }
    if (FACTORS) {
        if (tid > 0) params[6 + tid] = sqrt(sc / (tid == 1 ? ebeam : eext));
    } else {
        params[tid] = sc;
        params[3 + tid] = gc / sc;
        if (tid == 0) params[6] = M[(int64_t)g.nphi * g.theta_back] * 4 * PI_R4 / (g.waveno * g.waveno);
    }
}

}  // namespace abt

// Device epilogue.  ab/ae: amplitudes (8*nbins doubles, scaled by k in place), M: 3*16*nbins (total, beam,
// ext), m1d: 3*16*ntheta, params: 9 doubles.
extern "C" int abt_launch_finalise(const abt::DevGrid* g, double* ab, double* ae, double* M, double* m1d,
                                   double* params, int scaling, double ebeam, double eext, hipStream_t st)
{
    using namespace abt;
    // a lane per phi; whole waves, at most four
    const dim3 grid((unsigned)g->ntheta), block((unsigned)(g->nphi >= MB ? MB : (g->nphi + 63) / 64 * 64));
    const double* f = nullptr;
    if (scaling) {
        hipLaunchKernelGGL(k_epilogue<false>, grid, block, 0, st, *g, ab, ae, f, M, m1d);
        hipLaunchKernelGGL(k_theta_params<true>, dim3(1), dim3(MB), 0, st, *g, (const double*)m1d, (const double*)M,
                           ebeam, eext, params);
        f = params + 7;
    }
    hipLaunchKernelGGL(k_epilogue<true>, grid, block, 0, st, *g, ab, ae, f, M, m1d);
    hipLaunchKernelGGL(k_theta_params<false>, dim3(1), dim3(MB), 0, st, *g, (const double*)m1d, (const double*)M, ebeam,
                       eext, params);
    return (int)hipGetLastError();
}

// ---------------------------------------------------------------------------
// The epilogue without allocation (abt_finalise_dev_static).  Its limit is the entry point's: it once kept
// the total amplitude and the theta integrands (8 doubles per bin, 3 per theta) in a 64 MiB array.
static constexpr int64_t STATIC_SCRATCH_DOUBLES = (int64_t)8 << 20;

extern "C" int64_t abt_finalise_static_max_bins(int64_t n_theta)
{
    return n_theta < 0 ? 0 : (STATIC_SCRATCH_DOUBLES - 3 * n_theta) / 8;
}

extern "C" int abt_finalise_dev_static(const abt_dev_grid* g, double* ab, double* ae, int scaling,
                                       double ebeam, double eext, double* dev_mueller, double* dev_m1d,
                                       double* dev_params, void* stream)
{
    if (!g || !ab || !ae || !dev_mueller || !dev_m1d || !dev_params)
        return abt_fail(ABT_ERR_ARG, "abt_finalise_dev_static: null argument");
    if (g->d.nphi < 3 || g->d.ntheta < 3)
        return abt_fail(ABT_ERR_ARG, "finalise needs at least 3 theta and 3 phi values (simpne)");
    if (scaling && !(ebeam > 0 && eext > 0))
        return abt_fail(ABT_ERR_ARG, "energy scaling needs positive beam and ext energies");
    const int64_t need = 8 * (int64_t)g->nbins + 3 * (int64_t)g->d.ntheta;
    if (need > STATIC_SCRATCH_DOUBLES)
        return abt_fail(ABT_ERR_ARG,
                        "abt_finalise_dev_static: %lld bins x %d theta need %lld scratch doubles, more than the "
                        "%lld it holds (at most %lld bins at this theta count); use abt_finalise_dev",
                        (long long)g->nbins, g->d.ntheta, (long long)need, (long long)STATIC_SCRATCH_DOUBLES,
                        (long long)abt_finalise_static_max_bins(g->d.ntheta));
    int rc = abt_ensure_device(nullptr);
    if (rc) return rc;
    int e = abt_launch_finalise(&g->d, ab, ae, dev_mueller, dev_m1d, dev_params, scaling, ebeam, eext,
                                (hipStream_t)stream);
    if (e) return abt_fail(ABT_ERR_HIP, "finalise launch failed: %s", hipGetErrorString((hipError_t)e));
    return 0;
}
