// qsim_split_dev.h -- what the split-operator kernels of every length share:
// the device-side job description, the factor products and the 1D phase
// program.
#pragma once

#include "qsim_common.h"

namespace qsim {

enum { SW_FIRST = 0, SW_MID = 1, SW_LAST = 2 };

// Device-side description of one job (the kernels index a table of these by
// blockIdx.y, so many same-shape jobs share one launch).
struct SplitDev {
    c128 *psi;             // caller's complex128 state
    void *work;            // working state (== psi for precision 64)
    const c128 *ev[4];     // potential factors over the grid
    const c128 *kx[2];     // kinetic factor along x (2D) or the whole line (1D)
    const c128 *ky[2];     // kinetic factor along y (2D)
};

// v * f with f an FP64 factor.  FP32 data is widened, multiplied in FP64 and
// rounded once, so a near-identity factor (tiny V dt) keeps its sub-ulp part
// instead of losing it the same way at every step.  A float-float product
// that rounded v * hi before adding v * lo lost it: at 2048^2, dt = 0.1, that
// bias was half of a 1.1e-5 psi error after 1000 steps.
__device__ __forceinline__ c128 apply(c128 v, c128 f) { return v * f; }
__device__ __forceinline__ c64 apply(c64 v, c128 f) { return cvt<float>(cvt<double>(v) * f); }

// Phase program: start with ev[ev0]; each step runs (kinetic k[i], potential
// ev[e[i]]) for i < nph; the last potential factor of the last step is
// ev[ev_end] instead.
struct Prog1D {
    int ev0, ev_end, nph;
    int k[3], e[3];
};

}  // namespace qsim
