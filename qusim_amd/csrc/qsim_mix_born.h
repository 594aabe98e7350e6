// qsim_mix_born.h -- Born-series passes over mixed-radix lines (complex128).
#pragma once

#include "qsim_born_dev.h"
#include "qsim_mix.h"

namespace qsim {

// Workgroups per energy of the inner sweep; BornDev::resid holds 4 doubles for
// each.
size_t mix_born_blocks(const MixPlan &p, const BornGeom &geo);
// Inner sweep over the last axis (mode BA_START, BA_END or BA_BOTH) of the
// `nact` energies of `tab`.
int mix_born_inner(int mode, int pre, const BornDev *tab, int nact, const c128 *V,
                   const BornGeom &geo, const MixPlan &p, const void *tw, hipStream_t s);
// Outer sweep over axis 0: transform, G0, inverse transform.
int mix_born_outer(const BornDev *tab, int nact, const BornGeom &geo, const MixPlan &p,
                   const void *tw, hipStream_t s);
// Middle axis (3D): transform of tmp in place.
int mix_born_mid(bool inv, const BornDev *tab, int nact, const BornGeom &geo, const MixPlan &p,
                 const void *tw, hipStream_t s);
// out[2 a], out[2 a + 1]: residual and norm sums of the active energy a.
int mix_born_resid(const BornDev *tab, int nact, size_t nb, double *out, hipStream_t s);

}  // namespace qsim
