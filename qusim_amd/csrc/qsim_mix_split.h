// qsim_mix_split.h -- split-operator sweeps over mixed-radix lines.
#pragma once

#include "qsim_mix.h"
#include "qsim_split_dev.h"

namespace qsim {

// Row sweep (mode SW_FIRST / SW_MID / SW_LAST) of `nrows` rows of p.n points;
// SW_MID applies the potential factor `iev` once or twice.
int mix_row_sweep(int mode, const SplitDev &job, size_t nrows, int iev, bool twice,
                  const MixPlan &p, const void *tw, hipStream_t s);
// Column sweep of `ncols` columns of p.n points, stride ncols.
int mix_col_sweep(const SplitDev &job, size_t ncols, int ik, const MixPlan &p, const void *tw,
                  hipStream_t s);
// All steps of a 1D job in one workgroup.  nreal = p.n: a periodic line.
// nreal = p.n / 2: an infinite wall, run as the odd extension to p.n points
// (the job's factor tables are extended the same way, zero at 0 and nreal).
int mix_run_1d(const SplitDev &job, const Prog1D &prog, size_t nsteps, const MixPlan &p,
               size_t nreal, const void *tw, hipStream_t s);

}  // namespace qsim
