// Host check of the lengths that mix_plan (qsim_mix.h) refuses: a refused plan
// is empty (n = 0, what the dispatchers test), whatever the caller's MixPlan
// held before, and the set of refused lengths is the one that the LDS
// arithmetic gives: no composite of 2, 3, 5, 7, 11 and 13, and either no
// larger prime factor, or a line that with its twiddles does not fit 160 KiB
// twice.  Lengths given as arguments must be refused as well (the ones that
// the GPU tests take for the generic kernel and the unfused order).
// Prints one line per failure and "refused plans ok" when none fail.
#include <cstdio>
#include <cstdlib>

#include "qsim_fft_kernels.h"
#include "qsim_mix.h"

using namespace qsim;

static int failures = 0;

// the largest prime factor, and the number of prime factors up to 13
static void factors(int n, int *largest, int *small)
{
    *largest = 1;
    *small = 0;
    for (int p = 2; n > 1; ++p)
        while (n % p == 0) {
            *largest = p;
            *small += p <= 13;
            n /= p;
        }
}

// two lines of n elements with one of padding per 8, and the twiddles that
// the plan's passes index: (R - 1)(ns - 1) n / (ns R) + 1 of a pass and
// (P - 1) n / P + 1 of a prime's
static bool two_lines_fit(const MixPlan &p, int n)
{
    int tlen = 0;
    for (int dir = 0; dir < 2; ++dir)
        for (int i = 0; i < p.nf; ++i) {
            const MixPass &f = p.f[dir * kMixMaxPasses + i];
            const int a = (f.R - 1) * (f.ns - 1) * (n / (f.ns * f.R)) + 1;
            const int b = f.R > 15 ? (f.R - 1) * (n / f.R) + 1 : 0;
            if (a > tlen) tlen = a;
            if (b > tlen) tlen = b;
        }
    return 16 * (tlen + 2 * (n + n / 8)) <= 160 * 1024;
}

int main(int argc, char **argv)
{
    int refused = 0;
    for (int nw = 0; nw < 2 * (kMixMaxLen + 400); ++nw) {
        const int n = nw / 2;
        const double work = nw % 2 ? 8192 : n;
        MixPlan p;
        p.n = 77;   // a caller's earlier plan
        const bool ok = mix_plan(n, work, &p);
        if (!ok && p.n != 0) {
            std::printf("n=%d: refused, but the plan says n = %d\n", n, p.n);
            ++failures;
        }
        if (ok && p.n != n) {
            std::printf("n=%d: taken, but the plan says n = %d\n", n, p.n);
            ++failures;
        }
        refused += !ok && n >= 4 && n <= kMixMaxLen;
        if (n < 4) {
            failures += ok;
            continue;
        }
        int largest, small;
        factors(n, &largest, &small);
        bool want = n <= kMixMaxLen && (largest > 13 || small >= 2);
        if (ok && largest > 13) want = want && two_lines_fit(p, n);
        // no plan indexes more than n twiddles: refused only where those and
        // two lines do not fit
        if (!ok && largest > 13 && n <= kMixMaxLen)
            want = 16 * (n + 2 * (n + n / 8)) <= 160 * 1024;
        if (ok != want) {
            std::printf("n=%d: planned %d\n", n, ok);
            ++failures;
        }
    }
    for (int i = 1; i < argc; ++i) {
        const int n = std::atoi(argv[i]);
        if (n < 1) ++failures;
        for (double work : {(double)n, 8192.0}) {
            MixPlan p;
            if (mix_plan(n, work, &p)) {
                std::printf("n=%d: taken\n", n);
                ++failures;
            }
        }
    }
    std::printf("%d refused\n", refused / 2);
    if (!failures) std::printf("refused plans ok\n");
    return failures != 0;
}
