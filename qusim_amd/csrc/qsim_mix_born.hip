// qsim_mix_born.hip -- Born-series passes on mixed-radix lines: the fused
// schedule of qsim_born.hip for complex128 grids whose axes are not powers of
// two (inner sweep with the update and the next source, middle transforms,
// outer sweep with G0; every energy of the job in each launch).  An iteration
// of a 96^3 grid moves 176 B per point in 4 passes, 42 us an energy; the
// unfused order took 11 launches, 300 B and two synchronising reductions per
// energy: 285 us, 150 us with its transforms on mixed-radix lines.
#include "qsim_fft_kernels.h"
#include "qsim_mix_born.h"
#include "qsim_reduce.h"

namespace qsim {

using red::dd;
using red::dd_add;

__device__ __forceinline__ dd shfl_xor(dd a, int off)
{
    return dd{__shfl_xor(a.hi, off), __shfl_xor(a.lo, off)};
}

// MODE: BA_START, BA_END or BA_BOTH; PRE as in BornDev's jobs.  The sums of
// |new - old|^2 and |new|^2 are double-double throughout.
template <int MODE, int PRE>
__global__ void __launch_bounds__(kMixMaxThreads)
    k_mix_born_inner(const BornDev *__restrict__ jobs, const c128 *__restrict__ V, BornGeom geo,
                     MixPlan p, MixDims d, const c128 *__restrict__ tw)
{
    extern __shared__ unsigned char smem_raw[];
    MixWg<double> w = mix_begin<double>(smem_raw, p, d, tw);
    const BornDev &J = jobs[blockIdx.y];
    const unsigned nlines = (unsigned)(geo.n0 * geo.nmid), nmid = (unsigned)geo.nmid;
    const unsigned g = (blockIdx.x << d.logl) + (w.tid & ((1 << d.logl) - 1));
    const bool active = g < nlines;
    const unsigned gg = active ? g : 0, i = gg / nmid, j = gg % nmid;
    const size_t base = (size_t)gg * (unsigned)p.n;
    const int dim = geo.dim;
    c128 *tmp = reinterpret_cast<c128 *>(J.tmp) + base;
    c128 *dp = reinterpret_cast<c128 *>(J.dpsi) + base;
    V += base;
    // the separable tables: per-line factors, and the last axis's
    const double ab_line = dim == 3 ? ld_g(J.ab[0] + i) + ld_g(J.ab[1] + j) : ld_g(J.ab[0] + i);
    const c128 pw_line = dim == 3 ? ld_g(J.pw[0] + i) * ld_g(J.pw[1] + j) : ld_g(J.pw[0] + i);
    const double *ab_in = J.ab[dim == 3 ? 2 : 1];
    const c128 *pw_in = J.pw[dim == 3 ? 2 : 1];
    const double eps = J.eps, slow = J.slow, inv_eps = J.inv_eps, inv_n = J.inv_n;
    dd rsum{0, 0}, nsum{0, 0};

    auto keep = [](int, int, c128 v, c128) { return v; };
    if constexpr (MODE != BA_START) {
        mix_pass<MIX_FIRST>(w, p.f[0], MixNoPre(), [&](int, int m, c128, c128) {
            return mix_swap(ld_g(tmp + (unsigned)m));
        });
        for (int k = 1; k < p.nf; ++k) mix_pass<MIX_MID>(w, p.f[k], MixNoPre(), keep);
    }
    // The update and the next source, element by element in LDS: between the
    // transforms in registers (as the split sweeps' factors) the five arrays'
    // values of a whole butterfly spilled 550 B per lane.
    const int lm = (1 << d.logl) - 1, total = p.n << d.logl;
#pragma unroll 2
    for (int e = w.tid; e < total; e += d.nt) {
        const unsigned m = (unsigned)e >> d.logl;
        const c128 vk = ld_g(V + m);
        c128 o = ld_g(dp + m);
        const c128 ve =
            PRE == PRE_NAIVE ? vk : mk(vk.x, vk.y + (ab_line + ld_g(ab_in + m)));
        if constexpr (MODE != BA_START) {
            const c128 t = mix_swap(mix_ld(w, e & lm, (int)m)) * inv_n;
            const c128 nd = update<PRE>(o, t, ve, slow, eps, inv_eps);
            if (active) {
                store_nt(dp + m, nd);
                rsum = dd_add(rsum, abs2(nd - o));
                nsum = dd_add(nsum, abs2(nd));
            }
            o = nd;
        }
        if constexpr (MODE != BA_END) {
            const c128 s = source<PRE>(o, pw_line * ld_g(pw_in + m), ve, eps);
            w.lds[mix_slot(e, w.sh)] = s;
        }
    }
    if constexpr (MODE != BA_END) {
        if constexpr (MODE == BA_START) mix_wait_table();
        __syncthreads();
        mix_pass<MIX_HEAD>(w, p.f[0], MixNoPre(), keep);
        mix_inner(w, p, false);
        mix_pass<MIX_LAST>(w, mix_last(p, false), MixNoPre(), [&](int, int m, c128 v, c128) {
            if (active) store_nt(tmp + (unsigned)m, v);
            return v;
        });
    }
    if constexpr (MODE != BA_START) {
        // workgroup sums, over the LDS of the lines
        for (int off = 32; off > 0; off >>= 1) {
            rsum = dd_add(rsum, shfl_xor(rsum, off));
            nsum = dd_add(nsum, shfl_xor(nsum, off));
        }
        dd *slots = reinterpret_cast<dd *>(smem_raw);
        __syncthreads();
        if ((w.tid & 63) == 0) {
            slots[w.tid / 64 * 2] = rsum;
            slots[w.tid / 64 * 2 + 1] = nsum;
        }
        __syncthreads();
        if (w.tid == 0) {
            for (int k = 1; k < d.nt / 64; ++k) {
                rsum = dd_add(rsum, slots[2 * k]);
                nsum = dd_add(nsum, slots[2 * k + 1]);
            }
            double *o = J.resid + 4 * (size_t)blockIdx.x;
            o[0] = rsum.hi;
            o[1] = rsum.lo;
            o[2] = nsum.hi;
            o[3] = nsum.lo;
        }
    }
}

// G0 by Smith's division without its branch (op_G02D / op_G03D).
__device__ __forceinline__ c128 div_g0(c128 a, double wr, double wi)
{
    const bool big = fabs(wr) >= fabs(wi);
    const double p = big ? wr : wi, q = big ? wi : wr, r = q / p, den = p + q * r;
    const double x = big ? a.x + a.y * r : a.x * r + a.y;
    const double y = big ? a.y - a.x * r : a.y * r - a.x;
    return mk(x / den, y / den);
}

__global__ void __launch_bounds__(kMixMaxThreads)
    k_mix_born_outer(const BornDev *__restrict__ jobs, BornGeom geo, MixPlan p, MixDims d,
                     const c128 *__restrict__ tw)
{
    extern __shared__ unsigned char smem_raw[];
    MixWg<double> w = mix_begin<double>(smem_raw, p, d, tw);
    const BornDev &J = jobs[blockIdx.y];
    const unsigned S = (unsigned)(geo.n1 * geo.n2), n1 = (unsigned)geo.n1, n2 = (unsigned)geo.n2;
    const unsigned g = ((unsigned)xcd_tile(blockIdx.x, d.blocks) << d.logl) +
                       (w.tid & ((1 << d.logl) - 1));
    const bool active = g < S;
    const unsigned c = active ? g : 0;
    c128 *tmp = reinterpret_cast<c128 *>(J.tmp) + c;
    const int dim = geo.dim;
    const double fj = (double)fold_half(dim == 3 ? c / n2 : c, n1);
    const double fk = dim == 3 ? (double)fold_half(c % n2, n2) : 0.0;
    const double a0 = J.a[0], a1 = J.a[1], a2 = J.a[2], E = J.E, eps = J.eps;
    auto at = [&](int m) { return tmp + (size_t)(unsigned)m * S; };
    mix_two(
        w, p, [&](int, int m, c128, c128) { return ld_g(at(m)); }, MixNoPre(),
        [&](int, int m, c128 v, c128) {
            const double fi = (double)fold_half((size_t)m, (size_t)p.n);
            const double t = dim == 3 ? fi * fi * a0 + fj * fj * a1 + fk * fk * a2
                                      : fi * fi * a0 + fj * fj * a1;
            return mix_swap(div_g0(v, E - t, eps));
        },
        [&](int, int m, c128 v, c128) {
            if (active) store_nt(at(m), mix_swap(v));
            return v;
        });
}

template <bool INV>
__global__ void __launch_bounds__(kMixMaxThreads)
    k_mix_born_mid(const BornDev *__restrict__ jobs, BornGeom geo, MixPlan p, MixDims d,
                   const c128 *__restrict__ tw)
{
    extern __shared__ unsigned char smem_raw[];
    MixWg<double> w = mix_begin<double>(smem_raw, p, d, tw);
    const unsigned S = (unsigned)geo.n2, nlines = (unsigned)(geo.n0 * geo.n2);
    const unsigned g = ((unsigned)xcd_tile(blockIdx.x, d.blocks) << d.logl) +
                       (w.tid & ((1 << d.logl) - 1));
    const bool active = g < nlines;
    const unsigned gg = active ? g : 0;
    c128 *tmp = reinterpret_cast<c128 *>(jobs[blockIdx.y].tmp) +
                ((size_t)(gg / S) * (unsigned)p.n * S + gg % S);
    auto at = [&](int m) { return tmp + (size_t)(unsigned)m * S; };
    mix_one(
        w, p,
        [&](int, int m, c128, c128) {
            const c128 v = ld_g(at(m));
            return INV ? mix_swap(v) : v;
        },
        MixNoPre(),
        [&](int, int m, c128 v, c128) {
            if (active) store_nt(at(m), INV ? mix_swap(v) : v);
            return v;
        });
}

// One workgroup per energy adds the workgroups' sums in a fixed order.
__global__ void __launch_bounds__(256)
    k_mix_born_resid(const BornDev *__restrict__ tab, unsigned nb, double *__restrict__ out)
{
    __shared__ dd sh[2][256];
    const double *p = tab[blockIdx.x].resid;
    dd r{0, 0}, n{0, 0};
    for (unsigned b = threadIdx.x; b < nb; b += 256) {
        r = dd_add(r, dd{p[4 * (size_t)b], p[4 * (size_t)b + 1]});
        n = dd_add(n, dd{p[4 * (size_t)b + 2], p[4 * (size_t)b + 3]});
    }
    sh[0][threadIdx.x] = r;
    sh[1][threadIdx.x] = n;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
            for (int q = 0; q < 2; ++q)
                sh[q][threadIdx.x] = dd_add(sh[q][threadIdx.x], sh[q][threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x < 2)
        out[2 * blockIdx.x + threadIdx.x] = sh[threadIdx.x][0].hi + sh[threadIdx.x][0].lo;
}

// The launch shape is that of one energy, whatever shares the launch, so an
// energy's residual sums are the same alone and among others.
static MixShape inner_shape(const MixPlan &p, const BornGeom &geo)
{
    return mix_shape(p, geo.n0 * geo.nmid, sizeof(c128), false);
}
static MixShape strided_shape(const MixPlan &p, size_t nlines, int nact)
{
    MixShape sh = mix_shape(p, nlines * nact, sizeof(c128), true);
    sh.d.blocks = (unsigned)((nlines + ((size_t)1 << sh.d.logl) - 1) >> sh.d.logl);
    return sh;
}

size_t mix_born_blocks(const MixPlan &p, const BornGeom &geo)
{
    return inner_shape(p, geo).d.blocks;
}

template <int MODE, int PRE>
static int launch_inner(const BornDev *tab, int nact, const c128 *V, const BornGeom &geo,
                        const MixPlan &p, const void *tw, hipStream_t s)
{
    const MixShape sh = inner_shape(p, geo);
    auto fn = k_mix_born_inner<MODE, PRE>;
    QSIM_TRY(lds_limit((const void *)fn, kMixMaxLds));
    hipLaunchKernelGGL(fn, dim3(sh.d.blocks, (unsigned)nact), dim3(sh.d.nt), sh.lds, s, tab, V,
                       geo, p, sh.d, (const c128 *)tw);
    QSIM_HIP(hipGetLastError());
    return QSIM_OK;
}

template <int PRE>
static int inner_pre(int mode, const BornDev *tab, int nact, const c128 *V,
                     const BornGeom &geo, const MixPlan &p, const void *tw, hipStream_t s)
{
    // the source has two forms only
    constexpr int SRC = PRE == PRE_NAIVE ? PRE_NAIVE : PRE_IDENTITY;
    if (mode == BA_START) return launch_inner<BA_START, SRC>(tab, nact, V, geo, p, tw, s);
    if (mode == BA_END) return launch_inner<BA_END, PRE>(tab, nact, V, geo, p, tw, s);
    return launch_inner<BA_BOTH, PRE>(tab, nact, V, geo, p, tw, s);
}

int mix_born_inner(int mode, int pre, const BornDev *tab, int nact, const c128 *V,
                   const BornGeom &geo, const MixPlan &p, const void *tw, hipStream_t s)
{
    switch (pre) {
        case PRE_IDENTITY: return inner_pre<PRE_IDENTITY>(mode, tab, nact, V, geo, p, tw, s);
        case PRE_VELLEKOOP: return inner_pre<PRE_VELLEKOOP>(mode, tab, nact, V, geo, p, tw, s);
        case PRE_HAO1: return inner_pre<PRE_HAO1>(mode, tab, nact, V, geo, p, tw, s);
        case PRE_HAO2: return inner_pre<PRE_HAO2>(mode, tab, nact, V, geo, p, tw, s);
        default: return inner_pre<PRE_NAIVE>(mode, tab, nact, V, geo, p, tw, s);
    }
}

int mix_born_outer(const BornDev *tab, int nact, const BornGeom &geo, const MixPlan &p,
                   const void *tw, hipStream_t s)
{
    const MixShape sh = strided_shape(p, geo.n1 * geo.n2, nact);
    QSIM_TRY(lds_limit((const void *)k_mix_born_outer, kMixMaxLds));
    hipLaunchKernelGGL(k_mix_born_outer, dim3(sh.d.blocks, (unsigned)nact), dim3(sh.d.nt), sh.lds,
                       s, tab, geo, p, sh.d, (const c128 *)tw);
    QSIM_HIP(hipGetLastError());
    return QSIM_OK;
}

int mix_born_mid(bool inv, const BornDev *tab, int nact, const BornGeom &geo, const MixPlan &p,
                 const void *tw, hipStream_t s)
{
    const MixShape sh = strided_shape(p, geo.n0 * geo.n2, nact);
    auto fn = inv ? k_mix_born_mid<true> : k_mix_born_mid<false>;
    QSIM_TRY(lds_limit((const void *)fn, kMixMaxLds));
    hipLaunchKernelGGL(fn, dim3(sh.d.blocks, (unsigned)nact), dim3(sh.d.nt), sh.lds, s, tab, geo,
                       p, sh.d, (const c128 *)tw);
    QSIM_HIP(hipGetLastError());
    return QSIM_OK;
}

int mix_born_resid(const BornDev *tab, int nact, size_t nb, double *out, hipStream_t s)
{
    hipLaunchKernelGGL(k_mix_born_resid, dim3((unsigned)nact), dim3(256), 0, s, tab, (unsigned)nb,
                       out);
    QSIM_HIP(hipGetLastError());
    return QSIM_OK;
}

}  // namespace qsim
