// batch.h -- launch arguments of the orientation-batched far field (batch.hip), shared with
// its host plan (batch_plan.cpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sweep.h"

namespace abt {

// The epilogue of a group of consecutive orientations, o0 .. o1 - 1.
struct CombineArgs {
    DevGrid g;
    const double* part;       // [segment][8][nbins] segment sums of the group (SweepArgs::part)
    const double* ipart_inc;  // [segment][nbins] incoherent sums, or null
    const int32_t* seg_off;   // [2 norient + 1]: orientation o's beam-tree segments from 2o, ext tree's from 2o + 1
    const double* w1;         // [nbins] integral weights
    const double* w2;
    double* mpart;            // [nchunks][16][nbins] Mueller sums, or null (-scaling: formed later)
    double* ipart;            // [norient][ntiles][6] partial integrals
    double* ampl_out;         // [norient][8][nbins] k-scaled total amplitude per orientation, or null
    double* store;            // [norient][16][nbins] k-scaled beam then ext amplitude, or null
    double* epart;            // [nchunks][nbins] sums of S11_o * I_o (I_o: incoherent beam sum), or null
    const int32_t* list;      // list mode: the bins recomputed in FP64, ascending
    const int32_t* list_count;
    int o0, o1, nchunks, first;   // first: the chunk sums are stored, not added to
    int summed;               // each tree's segments are already summed, in its first
};

// A run's launches: groups of orientations whose segment sums fit the plan's buffer.
struct BatchGroup {
    int o0, o1;               // orientations
    int s0, s1;               // segments
};

struct BatchRun {
    SweepArgs sweep;          // segs: the plan's whole table
    CombineArgs comb;         // part, mpart, ...: the plan's buffers
    const BatchGroup* groups; // host
    int ngroups;
    int prec, tb, bpt;        // kernel precision and tile shape of the sweep
    int norient;              // orientations of this run (the autotuner's sample is a prefix)
    int nchunks;              // Mueller partial sums (1: summed in the output itself)
    double* mpart;            // [nchunks][16][nbins] when nchunks > 1
    const double* wphi;       // [nphi] weights of the phi integral
    double* mueller;
    double* mueller_1d;       // may be null
    double* integrals;
    hipStream_t st;
};

// Gated mixed precision: error-scale sums and scale, flags, the list of FP64 bins.
struct GateBufs {
    double* epart;            // [nchunks][nbins]
    double* est;              // [nbins]
    int32_t* flags;
    int32_t* list;
    int32_t* count;
    double* lpart;            // [nchunks][16][nbins] Mueller sums of the listed bins
};

// -scaling: the stored amplitudes, unscaled integrals and divisors, and the caller's energies.
struct ScaleBufs {
    double* store;            // [norient][16][nbins]
    double* raw;              // [norient][6]
    double* div;              // [norient][2]
    const double* beam_energy;
    const double* ext_energy;
};

}  // namespace abt

// The sweeps and epilogues of every group, the chunk and tile reductions, and (mueller_1d non-null)
// the phi integral of the summed matrix.
extern "C" int abt_launch_batch(const abt::BatchRun* r);
// -scaling (outputs_mod.f90:146-184): every orientation's beam and ext amplitudes stored, the unscaled
// integrals reduced into raw, the divisors sqrt(scatt_beam / beam_energy[o]) and sqrt(scatt_ext /
// ext_energy[o]) into div, the Mueller sums and all six integrals recomputed from the divided
// amplitudes, then the reductions.  ampl_out (non-null) receives the divided totals.
extern "C" int abt_launch_batch_scaled(const abt::BatchRun* r, const abt::ScaleBufs* s);
// Gated mixed precision: the mixed pass with its error scale, the bins whose error bound exceeds the
// gate listed, those bins recomputed in FP64 by the restructured body and written over the mixed
// pass's sums, then the phi integral.
extern "C" int abt_launch_batch_gated(const abt::BatchRun* r, const abt::GateBufs* q);
// The mixed pass of a gated plan alone (the autotuner's timing).
extern "C" int abt_launch_batch_est(const abt::BatchRun* r, const abt::GateBufs* q);
