// Host check of twiddle_powers (qsim_fft_core.h): over all first powers of
// the tables of 64 to 4096 points, the mean square error of the powers must
// not exceed that of the recurrence w^r = w^(r-1) w, which the lines that
// hold one power at a time use.  Prints "twiddle powers ok" or what failed.
#include <cmath>
#include <cstdio>

#include "qsim_fft_core.h"

using namespace qsim;

template <int R>
static int check(int n)
{
    const long double pi = 3.141592653589793238462643383279502884L;
    long double e[2] = {0, 0};
    for (int m = 1; m < n / R; ++m) {
        const long double a = -2.0L * pi * m / n;
        c128 w[R], v = mk((double)cosl(a), (double)sinl(a));
        w[1] = v;
        twiddle_powers<R>(w);
        c128 p = v;
        for (int r = 2; r < R; ++r) {
            p = p * v;
            const long double c = cosl(a * r), s = sinl(a * r);
            e[0] += (w[r].x - c) * (w[r].x - c) + (w[r].y - s) * (w[r].y - s);
            e[1] += (p.x - c) * (p.x - c) + (p.y - s) * (p.y - s);
        }
    }
    if (e[0] <= e[1]) return 0;
    std::printf("n=%d radix %d: %Lg times the recurrence's error\n", n, R, sqrtl(e[0] / e[1]));
    return 1;
}

int main()
{
    int failures = 0;
    for (int n = 64; n <= 4096; n *= 2) failures += check<4>(n) + check<8>(n);
    if (!failures) std::printf("twiddle powers ok\n");
    return failures != 0;
}
