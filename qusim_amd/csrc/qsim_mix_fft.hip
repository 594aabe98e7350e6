// qsim_mix_fft.hip -- mixed-radix transform of the lines of one tensor axis.
#include "qsim_fft_kernels.h"
#include "qsim_fft_plan.h"

namespace qsim {

// Lines of stride S (line_base), in -> out (in may be out: a workgroup reads
// all its lines before it stores any).  A 100 x 120 x 90 transform takes 3 x
// 10.6 us (35 MB a pass: 3.3 TB/s), with the generic kernel's sums over each
// factor 3 x 37 us.
template <typename T, bool INV>
__global__ void __launch_bounds__(kMixMaxThreads)
    k_fft_mix(const cx<T> *in, cx<T> *out, size_t S, size_t nlines,
              MixPlan p, MixDims d, const c128 *__restrict__ tw, double scale)
{
    extern __shared__ unsigned char smem_raw[];
    MixWg<T> w = mix_begin<T>(smem_raw, p, d, tw);
    const size_t g = (xcd_tile(blockIdx.x, d.blocks) << d.logl) + (w.tid & ((1 << d.logl) - 1));
    const bool active = g < nlines;
    const size_t base = active ? line_base(g, (size_t)p.n, S) : 0;
    in += base;
    out += base;
    mix_one(
        w, p,
        [&](int, int m, c128, c128) {
            const c128 v = cvt<double>(ld_g(in + (size_t)m * S));
            return INV ? mix_swap(v) : v;
        },
        MixNoPre(),
        [&](int, int m, c128 v, c128) {
            if (active) st_g(out + (size_t)m * S, cvt<T>((INV ? mix_swap(v) : v) * scale));
            return v;
        });
}

template <typename T, bool INV>
static int launch(const FftAxis &a, const void *in, void *out, double scale, hipStream_t s)
{
    const MixShape sh = mix_shape(a.mix, a.nlines, sizeof(cx<T>), a.S > 1);
    QSIM_CHECK(sh.d.nt > 0, "mixed-radix transform: launch shape");
    auto fn = k_fft_mix<T, INV>;
    QSIM_TRY(lds_limit((const void *)fn, kMixMaxLds));
    hipLaunchKernelGGL(fn, dim3(sh.d.blocks), dim3(sh.d.nt), sh.lds, s, (const cx<T> *)in,
                       (cx<T> *)out, a.S, a.nlines, a.mix, sh.d,
                       (const c128 *)a.tw, scale);
    QSIM_HIP(hipGetLastError());
    return QSIM_OK;
}

int launch_fft_mix(const FftAxis &a, int precision, bool inv, const void *in, void *out,
                   double scale, hipStream_t s)
{
    if (precision == 64)
        return inv ? launch<double, true>(a, in, out, scale, s)
                   : launch<double, false>(a, in, out, scale, s);
    return inv ? launch<float, true>(a, in, out, scale, s)
               : launch<float, false>(a, in, out, scale, s);
}

}  // namespace qsim
