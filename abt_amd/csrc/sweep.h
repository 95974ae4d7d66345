// sweep.h -- launch arguments of the beam sweep (far_field.hip): the coherent sums of beam
// segments on every bin, which the single-orientation far field (runtime.cpp) and the
// orientation-batched plan (batch.hip) build on.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "adjbody.h"
#include "ffbody.h"
#include "records.h"

namespace abt {

// A bin's complete beam sum to its amplitude matrix (temp_rot1, and the bin's far-field phase for
// the bodies that sum relative to it).  PREC: the kernel precision.
template <int PREC>
__device__ __forceinline__ void finish_sum(double acc[8], const DevGrid& g, int bin)
{
    const int iphi = bin % g.nphi;
    const double cp = g.cphi[iphi], sp = g.sphi[iphi];
    if (PREC == 0 || PREC == 1) mixed_finish(acc, cp, sp);
    if (PREC == 3) model_finish(acc, cp, sp, g.kr_rev[bin]);
    if (PREC == 4) fp64r_finish(acc, cp, sp, g.kr_rev[bin]);
}

// One beam segment of a batched plan: `count` consecutive records of one tree.
struct SweepSeg {
    int64_t start;    // first record (index into the tree's records)
    int32_t count;
    int32_t tree;     // 0: beam tree, 1: ext tree
};

struct SweepArgs {
    DevGrid g;
    const double* recs[2];    // prepared records of the beam and ext trees
    const double* vrecs[2];
    const SweepSeg* segs;     // [gridDim.y] segments, or null: segment s is records
    int64_t nb, per;          // s * per .. min(nb, (s + 1) * per) of tree 0
    double* part;             // [segment][8][nbins] segment sums as the body forms them, or null:
    double* out;              // the finished sum of the one segment (Fortran layout; PREC 2: [nbins])
    double* ipart;            // [segment][nbins] incoherent sums (INC)
    const int32_t* list;      // LIST: the bins of the lane slots
    const int32_t* list_count;
    int fast_diff;
};

// Sweep variants: plain, with the incoherent beam sum, over a list of bins.
enum : int { SWEEP_PLAIN = 0, SWEEP_INC = 1, SWEEP_LIST = 2 };

}  // namespace abt

// Kernel instance for (kernel precision, beams between barriers, bins per lane, variant); nullptr if none.
// Kernel precisions: 0 plain FP64, 1 mixed, 2 incoherent FP64, 3 frame-free FP64 model, 4 restructured FP64.
extern "C" const void* abt_sweep_kernel(int prec, int tb, int bpt, int mode);
extern "C" int abt_launch_sweep(const abt::SweepArgs* a, int nseg, int prec, int tb, int bpt, int mode,
                                hipStream_t st);
