// qsim_mix_split.hip -- split-operator sweeps whose lines are not a power of
// two (qsim_mix.h): the schedule of qsim_split.hip's fused jobs, on
// mixed-radix lines in complex128.  The factors are applied one by one as the
// unfused order does (the half step's factor twice where two half steps
// meet, 1/n apart from the kinetic factor): a product of two factors rounded
// once into a table repeats its rounding at every step.
#include "qsim_fft_kernels.h"
#include "qsim_mix_split.h"

namespace qsim {

constexpr int kMix1dThreads = 768;

// Lines are read once a sweep: from 6 MiB a sweep on, non-temporal loads keep
// E_V and the tables in L2.  us a step with plain and with non-temporal loads:
// 300 x 300 (1.4 MiB) 17.0 and 18.0, 500 x 500 (3.8) 21.4 and 21.7, 600 x 600
// (5.5) 24.4 and 24.5, 640 x 660 (6.4) 26.7 and 26.6, 700 x 700 (7.5) 28.3 and
// 27.8, 900 x 900 32.8 and 30.4, 1000 x 1000 35.5 and 31.9, 1500 x 1500 81.7 and
// 80.6.
template <bool NT>
__device__ __forceinline__ c128 ld_psi(const c128 *p)
{
    if constexpr (NT) return ld_nt(p);
    else return ld_g(p);
}
static bool psi_nt(const MixPlan &p, size_t nlines)
{
    return (size_t)p.n * nlines * sizeof(c128) >= ((size_t)6 << 20);
}

// Row and column sweeps: 32 B of psi and 16 B of E_V per point move once.  At
// 1000 x 1000 a step takes 32 us (the unfused order's 8 passes: 300 us) and at
// 1500 x 1500 80 us (2.2 TB/s of the 80 B); below that the chain of one
// workgroup's passes bounds the sweeps (750 x 600: 28 us a step, waves wait for
// 76% of their cycles in the row sweep and 65% in the column sweep), above it
// the LDS exchanges.
template <int MODE, bool NT>
__global__ void __launch_bounds__(kMixMaxThreads)
    k_mix_row(c128 *psi, const c128 *ev, int twice, unsigned nrows, MixPlan p, MixDims d,
              const c128 *__restrict__ tw)
{
    extern __shared__ unsigned char smem_raw[];
    MixWg<double> w = mix_begin<double>(smem_raw, p, d, tw);
    // every butterfly of a thread is on the same line (L divides the threads);
    // threads past the last line read line 0 and store nothing
    const unsigned g = (blockIdx.x << d.logl) + (w.tid & ((1 << d.logl) - 1));
    const bool active = g < nrows;
    const size_t base = (size_t)(active ? g : 0) * (unsigned)p.n;
    psi += base;
    ev += base;
    auto evm = [&](int, int m) { return ld_g(ev + (unsigned)m); };
    auto store = [&](int, int m, c128 v, c128) {
        if (active) store_nt(psi + (unsigned)m, v);
        return v;
    };
    auto load_inv = [&](int, int m, c128, c128) { return mix_swap(ld_psi<NT>(psi + (unsigned)m)); };
    if constexpr (MODE == SW_FIRST) {
        mix_one(
            w, p,
            [&](int, int m, c128, c128) {
                return ld_g(psi + (unsigned)m) * ld_g(ev + (unsigned)m);
            },
            MixNoPre(), store);
    } else if constexpr (MODE == SW_MID) {
        mix_two(
            w, p, load_inv, evm,
            [&](int, int, c128 v, c128 e) {
                v = mix_swap(v) * e;
                return twice ? v * e : v;
            },
            store);
    } else {
        mix_one(w, p, load_inv, evm, [&](int, int m, c128 v, c128 e) {
            if (active) store_nt(psi + (unsigned)m, mix_swap(v) * e);
            return v;
        });
    }
}

template <bool NT>
__global__ void __launch_bounds__(kMixMaxThreads)
    k_mix_col(c128 *psi, const c128 *kx, const c128 *ky, double scale, double scale_lo,
              unsigned ncols, MixPlan p, MixDims d, const c128 *__restrict__ tw)
{
    extern __shared__ unsigned char smem_raw[];
    MixWg<double> w = mix_begin<double>(smem_raw, p, d, tw);
    const unsigned g = ((unsigned)xcd_tile(blockIdx.x, d.blocks) << d.logl) +
                       (w.tid & ((1 << d.logl) - 1));
    const bool active = g < ncols;
    const unsigned c = active ? g : 0;
    psi += c;
    const c128 kyj = ld_g(ky + c);
    auto at = [&](int m) { return psi + (size_t)((unsigned)m * (size_t)ncols); };
    mix_two(
        w, p, [&](int, int m, c128, c128) { return ld_psi<NT>(at(m)); },
        [&](int, int m) { return ld_g(kx + (unsigned)m); },
        [&](int, int, c128 v, c128 k) { return mix_swap(v * k * kyj); },
        [&](int, int m, c128 v, c128) {
            if (active) store_nt(at(m), mix_scale(mix_swap(v), scale, scale_lo));
            return v;
        });
}

// All steps of one line: 768 threads at most, so that 168 registers are left (at
// 128 the wide radices spilled: 1000 points 6.2 against 5.3 us a step when
// timed).  Bound by the latency of its passes: a step of n = 1000 is 6 of about
// 1 us (an O4 stage 6.0 us); the unfused order's 7 launches took 66 us.
__global__ void __launch_bounds__(kMix1dThreads)
    k_mix_1d(SplitDev J, Prog1D prog, size_t nsteps, double scale, double scale_lo,
             MixPlan p, MixDims d, int nreal, const c128 *__restrict__ tw)
{
    extern __shared__ unsigned char smem_raw[];
    MixWg<double> w = mix_begin<double>(smem_raw, p, d, tw);
    c128 *psi = J.psi;
    const c128 *e0 = J.ev[prog.ev0];
    const bool wall = nreal != p.n;
    mix_pass<MIX_FIRST>(w, p.f[0], MixNoPre(), [&](int, int m, c128, c128) {
        if (wall && (m == 0 || m == nreal)) return mk(0.0, 0.0);
        const c128 v = ld_g(psi + (m < nreal ? m : p.n - m)) * ld_g(e0 + m);
        return m < nreal ? v : mk(-v.x, -v.y);
    });
    for (size_t st = 0; st < nsteps; ++st)
        for (int ph = 0; ph < prog.nph; ++ph) {
            const c128 *kt = J.kx[prog.k[ph]];
            const bool last = st + 1 == nsteps && ph + 1 == prog.nph;
            // between steps the closing and the opening half step meet
            const bool twice = ph + 1 == prog.nph;
            const c128 *ev = J.ev[last ? prog.ev_end : prog.e[ph]];
            mix_inner(w, p, false);
            mix_pass<MIX_TURN, 10>(
                w, mix_last(p, false), [&](int, int m) { return ld_g(kt + m); },
                [&](int, int, c128 v, c128 k) { return mix_swap(v * k); });
            mix_inner(w, p, true);
            auto evm = [&](int, int m) { return ld_g(ev + m); };
            if (last)
                mix_pass<MIX_LAST, 10>(w, mix_last(p, true), evm, [&](int, int m, c128 v, c128 e) {
                    if (m < nreal) st_g(psi + m, mix_scale(mix_swap(v), scale, scale_lo) * e);
                    return v;
                });
            else
                mix_pass<MIX_TURN, 10>(w, mix_last(p, true), evm, [&](int, int, c128 v, c128 e) {
                    v = mix_scale(mix_swap(v), scale, scale_lo) * e;
                    return twice ? v * e : v;
                });
        }
}

template <int MODE>
static int launch_row(const SplitDev &job, size_t nrows, int iev, bool twice,
                      const MixPlan &p, const void *tw, hipStream_t s)
{
    const MixShape sh = mix_shape(p, nrows, sizeof(c128), false);
    auto fn = k_mix_row<MODE, false>;
    if constexpr (MODE != SW_FIRST)
        if (psi_nt(p, nrows)) fn = k_mix_row<MODE, true>;
    QSIM_TRY(lds_limit((const void *)fn, kMixMaxLds));
    hipLaunchKernelGGL(fn, dim3(sh.d.blocks), dim3(sh.d.nt), sh.lds, s, job.psi,
                       job.ev[iev], (int)twice, (unsigned)nrows, p, sh.d, (const c128 *)tw);
    QSIM_HIP(hipGetLastError());
    return QSIM_OK;
}

int mix_row_sweep(int mode, const SplitDev &job, size_t nrows, int iev, bool twice,
                  const MixPlan &p, const void *tw, hipStream_t s)
{
    if (mode == SW_FIRST) return launch_row<SW_FIRST>(job, nrows, iev, twice, p, tw, s);
    if (mode == SW_MID) return launch_row<SW_MID>(job, nrows, iev, twice, p, tw, s);
    return launch_row<SW_LAST>(job, nrows, iev, twice, p, tw, s);
}

int mix_col_sweep(const SplitDev &job, size_t ncols, int ik, const MixPlan &p, const void *tw,
                  hipStream_t s)
{
    const MixShape sh = mix_shape(p, ncols, sizeof(c128), true);
    auto fn = psi_nt(p, ncols) ? k_mix_col<true> : k_mix_col<false>;
    QSIM_TRY(lds_limit((const void *)fn, kMixMaxLds));
    const double n = (double)p.n * (double)ncols;
    hipLaunchKernelGGL(fn, dim3(sh.d.blocks), dim3(sh.d.nt), sh.lds, s, job.psi,
                       job.kx[ik], job.ky[ik], 1.0 / n, mix_recip_lo(n), (unsigned)ncols, p,
                       sh.d, (const c128 *)tw);
    QSIM_HIP(hipGetLastError());
    return QSIM_OK;
}

int mix_run_1d(const SplitDev &job, const Prog1D &prog, size_t nsteps, const MixPlan &p,
               size_t nreal, const void *tw, hipStream_t s)
{
    const MixShape sh = mix_shape_of(p, 0, 1, sizeof(c128), kMixMaxLds);
    QSIM_CHECK(sh.d.nt > 0 && sh.d.nt <= kMix1dThreads, "1D line: launch shape");
    QSIM_TRY(lds_limit((const void *)k_mix_1d, kMixMaxLds));
    hipLaunchKernelGGL(k_mix_1d, dim3(1), dim3(sh.d.nt), sh.lds, s, job, prog, nsteps, 1.0 / p.n,
                       mix_recip_lo(p.n), p, sh.d, (int)nreal, (const c128 *)tw);
    QSIM_HIP(hipGetLastError());
    return QSIM_OK;
}

}  // namespace qsim
