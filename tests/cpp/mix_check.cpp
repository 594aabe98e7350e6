// Host check of the mixed-radix plans (qsim_mix.h): every length that
// mix_plan takes is run through its passes on the host, with the kernels' own
// butterflies, twiddles and index rules, in both radix orders, and compared
// with a long double DFT; the launch shapes must cover every butterfly of
// every pass within mix_k per thread and stay inside 160 KiB of LDS;
// the strided sweeps' tile order must be a permutation.
// Prints one line per failure and "mixed plans ok" when none fail.
#include <cmath>
#include <complex>
#include <cstdio>
#include <vector>

#include "qsim_fft_kernels.h"
#include "qsim_mix.h"

using namespace qsim;

static int failures = 0, tlen = 0;

template <int R>
static void pass_r(std::vector<c128> &x, const MixPass &p, const std::vector<c128> &tw)
{
    std::vector<c128> y(x.size());
    for (int j = 0; j < p.nb; ++j) {
        c128 v[R];
        for (int r = 0; r < R; ++r) v[r] = x[j + r * p.nb];
        const int k = mix_mod(p, j), base = (j - k) * R + k;
        if (p.ns > 1) {
            MixTw<R> t;
            if (k != j % p.ns || (R - 1) * k * p.tws >= tlen) {
                std::printf("n=%zu R=%d j=%d: index\n", x.size(), R, j);
                ++failures;
                return;
            }
            t.load(tw.data(), k * p.tws);
            t.dft(v);
        } else {
            mix_dft<R>(v);
        }
        for (int r = 0; r < R; ++r) y[base + r * p.ns] = v[r];
    }
    x.swap(y);
}

// a prime's pass through the kernels' own pair and output stages; every
// element must be written once
struct At {
    std::vector<c128> &x;
    c128 get(int e) const { return x.at(e); }
    void set(int e, c128 v) const { x.at(e) = v; }
};
template <int M>
static void prime_m(std::vector<c128> &x, const MixPass &p, const std::vector<c128> &tw)
{
    std::vector<c128> y(x.size());
    std::vector<int> hit(x.size(), 0);
    const int H = (p.R - 1) / 2;
    for (int j = 0; j < p.nb; ++j) {
        if ((p.R - 1) * mix_mod(p, j) * p.tws >= tlen || (p.R - 1) * p.nb >= tlen) ++failures;
        for (int k = 1; k <= H; ++k) mix_prime_pair(p, tw.data(), j, k, At{x});
    }
    const int dm = (H + M) / M;
    for (int j = 0; j < p.nb; ++j)
        for (int m = 0; m < dm; ++m)
            mix_prime_out<M>(p, tw.data(), j, m, dm, At{x}, [&](int e, c128 v) {
                y.at(e) = v;
                ++hit[e];
            });
    // the flat item index splits as the kernel splits it
    const unsigned mag = p.nb == 1 ? 0u : 0xffffffffu / (unsigned)p.nb + 1u;
    for (int t = 0; t < p.nb * (H + 1) && p.nb > 1; ++t)
        if ((int)mix_mulhi(t, mag) != t / p.nb) ++failures;
    for (int h : hit)
        if (h != 1) ++failures;
    x.swap(y);
}

static void prime(std::vector<c128> &x, const MixPass &p, const std::vector<c128> &tw)
{
    static int turn = 0;
    if (++turn % 3 == 0) prime_m<1>(x, p, tw);
    else if (turn % 3 == 1) prime_m<2>(x, p, tw);
    else prime_m<4>(x, p, tw);
}

static void transform(std::vector<c128> &x, const MixPass *f, int nf, const std::vector<c128> &tw)
{
    for (int i = 0; i < nf; ++i) switch (f[i].R) {
#define CASE(R_) case R_: pass_r<R_>(x, f[i], tw); break;
            CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11)
            CASE(12) CASE(13) CASE(14) CASE(15) CASE(1)
#undef CASE
            default: prime(x, f[i], tw);
        }
}

// 1: prime factors of at most 13 (two of them), 2: with larger ones, 0: neither
static int smooth(int n)
{
    int m = n, np = 0;
    for (int p : {2, 3, 5, 7, 11, 13})
        while (m % p == 0) m /= p, ++np;
    if (m == 1) return np >= 2 && n >= 4;
    for (int p = 17; p <= n; ++p)
        while (m % p == 0) m /= p;
    return m == 1 && n > 13 ? 2 : 0;
}

int main()
{
    const long double pi = 3.141592653589793238462643383279502884L;
    // the tiles of a strided sweep are dealt to the XCDs one to one
    for (size_t nb = 1; nb < 700; ++nb) {
        std::vector<int> hit(nb, 0);
        for (size_t b = 0; b < nb; ++b) {
            const size_t t = xcd_tile(b, nb);
            if (t >= nb || hit[t]++) {
                std::printf("xcd_tile(%zu, %zu) = %zu\n", b, nb, t);
                ++failures;
                break;
            }
        }
    }
    int planned = 0;
    for (int nw = 2; nw < 2 * (kMixMaxLen + 200); ++nw) {
        // every length as a line that a CU holds alone and among many
        const int n = nw / 2;
        MixPlan p;
        const bool ok = mix_plan(n, nw % 2 ? 8192 : n, &p);
        // lengths with a larger prime: all up to 3100 points (two lines in LDS)
        const int sm = smooth(n);
        if (sm == 2 && n > 3100 && !ok) continue;
        if (ok != (sm != 0 && n <= kMixMaxLen)) {
            std::printf("n=%d planned %d\n", n, ok);
            ++failures;
            continue;
        }
        if (!ok) continue;
        ++planned;
        int prod = 1;
        for (int i = 0; i < p.nf; ++i) {
            prod *= p.f[i].R;
            if (p.f[kMixMaxPasses + i].R != p.f[p.nf - 1 - i].R) ++failures;
        }
        if (prod != n || p.nf < 2) {
            std::printf("n=%d: radices\n", n);
            ++failures;
        }
        for (size_t lines : {1, 2, 7, 100, 600, 100000})
            for (int es : {8, 16})
                for (bool st : {false, true}) {
                    const MixShape s = mix_shape(p, lines, es, st);
                    const int L = 1 << s.d.logl;
                    bool bad = s.d.nt % 64 || s.d.nt < 64 || s.d.nt > kMixMaxThreads ||
                               s.d.nt % L || s.lds > 160 * 1024 ||
                               s.lds < p.tlen * sizeof(c128) + (s.d.alt + mix_slot(n * L - 1, s.d.sh) + 1) * (size_t)es ||
                               (s.d.alt && s.d.alt <= mix_slot(n * L - 1, s.d.sh)) ||
                               p.tlen > n || (size_t)s.d.blocks * L < lines ||
                               ((size_t)s.d.blocks - 1) * L >= lines;
                    for (int i = 0; i < p.nf; ++i)
                        bad = bad || (p.f[i].R <= 15 && p.f[i].nb * L > s.d.nt * mix_k(p.f[i].R));
                    bad = bad || (p.prime && !s.d.alt);
                    for (int i = 0; i < p.nf; ++i)   // primes in the middle
                        bad = bad || (p.f[i].R > 15 && (i == 0 || i == p.nf - 1));
                    // the 1D kernel runs one line on at most 768 threads
                    const MixShape one = mix_shape_of(p, 0, 1, 16, kMixMaxLds);
                    bad = bad || one.d.nt < 64 || one.d.nt > 768 || one.lds > kMixMaxLds;
                    if (bad) {
                        std::printf("n=%d lines=%zu es=%d strided=%d: launch shape\n", n, lines,
                                    es, st);
                        ++failures;
                    }
                }
        // the values: every length up to 260 and a spread of longer ones
        if (n > 260 && n % 50 && n % 143 && n % 64 && n != 2738 && n != 5005 && n != 323 &&
            n != 4913 && n != 2003)
            continue;
        std::vector<c128> tw(n), x(n);
        std::vector<std::complex<long double>> w(n);
        unsigned s = 12345u + n;
        for (int m = 0; m < n; ++m) {
            const long double a = -2.0L * pi * m / n;
            w[m] = {cosl(a), sinl(a)};
            tw[m] = mk((double)cosl(a), (double)sinl(a));
            s = s * 1664525u + 1013904223u;
            x[m].x = (s >> 8) / 8388608.0 - 1.0;
            s = s * 1664525u + 1013904223u;
            x[m].y = (s >> 8) / 8388608.0 - 1.0;
        }
        std::vector<c128> a = x, b = x;
        tlen = p.tlen;
        transform(a, p.f, p.nf, tw);
        transform(b, p.f + kMixMaxPasses, p.nf, tw);
        long double ea = 0, eb = 0, ref = 0;
        const int step = n > 1000 ? 37 : 1;   // spot check the longer lines
        for (int k = 0; k < n; k += step) {
            std::complex<long double> t = 0;
            for (int m = 0; m < n; ++m)
                t += std::complex<long double>(x[m].x, x[m].y) * w[(size_t)m * k % n];
            ea += std::norm(t - std::complex<long double>(a[k].x, a[k].y));
            eb += std::norm(t - std::complex<long double>(b[k].x, b[k].y));
            ref += std::norm(t);
        }
        // a pass adds a few units of 2^-53 per element, a prime's pass about
        // sqrt(P / 2) / 2 more; 6 passes stay below 32
        if (!(sqrtl(ea / ref) < 32 * 1.1102230246251565e-16L) ||
            !(sqrtl(eb / ref) < 32 * 1.1102230246251565e-16L)) {
            std::printf("n=%d: rel L2 %Lg and %Lg\n", n, sqrtl(ea / ref), sqrtl(eb / ref));
            ++failures;
        }
    }
    std::printf("%d lengths planned\n", planned);
    if (!failures) std::printf("mixed plans ok\n");
    return failures != 0;
}
