// qsim_born_dev.h -- what the Born-series kernels of every length share: the
// grid, the per-energy description and the pointwise stages.
#pragma once

#include "qsim_common.h"

namespace qsim {

enum { BA_START = 0, BA_END = 1, BA_BOTH = 2 };
enum { PRE_IDENTITY = 0, PRE_VELLEKOOP = 1, PRE_HAO1 = 2, PRE_HAO2 = 3, PRE_NAIVE = 4 };

struct BornGeom {
    int dim;
    size_t n0, n1, n2;   // n2 = 1 for 2D
    size_t ninner;       // length of the last axis
    size_t nmid;         // 3D: n1; 2D: 1
};

// per-energy device descriptor
struct BornDev {
    void *dpsi;
    void *tmp;
    const c128 *pw[3];     // plane-wave factor per axis: exp(i k_a x_a)
    const double *ab[3];   // absorbing-layer Im V per axis (zeros when naive)
    double E, eps, slow, inv_n;
    double inv_eps;        // 1 / eps (0 when eps is 0)
    double a[3];           // (2 pi hbar / (d n))^2 / 2m per axis
    double *resid;         // residual partial sums: 2 per block, on mixed-radix grids 4
};

// potential with the absorbing layer, in the reference's summation order
__device__ __forceinline__ c128 v_eff(c128 v, const BornDev &J, int dim, size_t i, size_t j,
                                      size_t k)
{
    const double a = dim == 3 ? (ld_g(J.ab[0] + i) + ld_g(J.ab[1] + j)) + ld_g(J.ab[2] + k)
                              : ld_g(J.ab[0] + i) + ld_g(J.ab[1] + j);
    return mk(v.x, v.y + a);
}

__device__ __forceinline__ c128 psi0_at(const BornDev &J, int dim, size_t i, size_t j, size_t k)
{
    return dim == 3 ? (ld_g(J.pw[0] + i) * ld_g(J.pw[1] + j)) * ld_g(J.pw[2] + k)
                    : ld_g(J.pw[0] + i) * ld_g(J.pw[1] + j);
}

// gamma of op_Vellekoop / op_Hao1 / op_Hao2 (src/DeviceTemplate.h:1020-1077)
// with the divisions by eps done as products with 1/eps: within an ulp of the
// quotient, without two FP64 divide sequences per point in the fused sweeps.
// op_Hao2's 2 / w, w = 1 + i v / eps = (1 - v.y / eps, v.x / eps), is taken
// as 2 conj(w) / |w|^2 with one real divide instead of a complex division
// (|w|^2 >= 1 for the absorbing potentials, Im v <= 0, so the unscaled form
// neither overflows nor underflows); that also frees the registers the
// merged plane pass needs.
template <int PRE>
__device__ __forceinline__ c128 gamma_fused(c128 v, double slow, double eps, double inv_eps)
{
    if constexpr (PRE == PRE_VELLEKOOP) {
        const c128 iv = imul(v);
        return mk(1. - iv.x * inv_eps, -iv.y * inv_eps) * slow;
    } else if constexpr (PRE == PRE_HAO1) {
        const c128 iv = imul(mk(v.x, -v.y));
        return mk(1. - iv.x * inv_eps, -iv.y * inv_eps) * slow;
    } else {
        const double wr = 1. - v.y * inv_eps, wi = v.x * inv_eps;
        const double s2 = 2. * slow / (wr * wr + wi * wi);
        return mk(wr * s2, -wi * s2);
    }
}

template <int PRE>
__device__ __forceinline__ c128 update(c128 dpsi, c128 t, c128 v, double slow, double eps,
                                       double inv_eps)
{
    if constexpr (PRE == PRE_NAIVE) {
        return t;
    } else if constexpr (PRE == PRE_IDENTITY) {
        return slow == 1. ? t : dpsi * (1 - slow) + t * slow;
    } else {
        c128 g = gamma_fused<PRE>(v, slow, eps, inv_eps);
        return mk(1. - g.x, -g.y) * dpsi + g * t;
    }
}

template <int PRE>
__device__ __forceinline__ c128 source(c128 dpsi, c128 p0, c128 v, double eps)
{
    if constexpr (PRE == PRE_NAIVE) return (dpsi + p0) * v;          // op_AddMul
    else return mk(v.x, v.y + eps) * dpsi + v.x * p0;                // op_Add3
}

}  // namespace qsim
