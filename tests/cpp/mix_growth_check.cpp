// Host check of how the mixed-radix transforms' error grows (qsim_mix.h, the
// kernels' own butterflies, twiddles and scaling): 60 steps of forward
// transform, phase factors, inverse transform in the reverse radix order and
// 1 / n, against long double, beside the same steps with direct sums of R
// table products per output (the generic kernel's order: radices 4, 2, 3, 5,
// 7, ...).  Rounded constants repeat their rounding every step, so their error
// grows with the steps; compensated ones leave it to the random roundings.
// Bounds: the ratio of the two errors at most 1 in the geometric mean over the
// lengths, for one transform and for the steps, and for the steps at most 1.2
// at every length (the factors of a length make its ratio vary by a fifth).
// Prints one line per failure and "error growth ok" when none fail.
#include <cmath>
#include <complex>
#include <cstdio>
#include <vector>

#include "qsim_fft_kernels.h"
#include "qsim_mix.h"

using namespace qsim;
using ld = long double;
using cl = std::complex<long double>;
using Line = std::vector<c128>;

static const ld kPi = 3.141592653589793238462643383279502884L;

template <int R>
static void pass_r(Line &x, const MixPass &p, const Line &tw)
{
    Line y(x.size());
    for (int j = 0; j < p.nb; ++j) {
        c128 v[R];
        for (int r = 0; r < R; ++r) v[r] = x[j + r * p.nb];
        const int k = mix_mod(p, j), base = (j - k) * R + k;
        if (p.ns > 1) {
            MixTw<R> t;
            t.load(tw.data(), k * p.tws);
            t.dft(v);
        } else {
            mix_dft<R>(v);
        }
        for (int r = 0; r < R; ++r) y[base + r * p.ns] = v[r];
    }
    x.swap(y);
}

struct At {
    Line &x;
    c128 get(int e) const { return x[e]; }
    void set(int e, c128 v) const { x[e] = v; }
};
static void prime(Line &x, const MixPass &p, const Line &tw)
{
    Line y(x.size());
    const int H = (p.R - 1) / 2;
    for (int j = 0; j < p.nb; ++j)
        for (int k = 1; k <= H; ++k) mix_prime_pair(p, tw.data(), j, k, At{x});
    for (int j = 0; j < p.nb; ++j)
        for (int m = 0; m <= H; ++m)
            mix_prime_out<1>(p, tw.data(), j, m, H + 1, At{x}, [&](int e, c128 v) { y[e] = v; });
    x.swap(y);
}

static void mixed(Line &x, const MixPass *f, int nf, const Line &tw)
{
    for (int i = 0; i < nf; ++i) switch (f[i].R) {
#define CASE(R_) case R_: pass_r<R_>(x, f[i], tw); break;
            CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10)
            CASE(11) CASE(12) CASE(13) CASE(14) CASE(15)
#undef CASE
            default: prime(x, f[i], tw);
        }
}

// a product with one rounding fewer, as the device compiles it
static c128 mul(c128 a, c128 b)
{
    return mk(std::fma(a.x, b.x, -(a.y * b.y)), std::fma(a.x, b.y, a.y * b.x));
}
static c128 conj(c128 a) { return mk(a.x, -a.y); }

static void direct(Line &x, const Line &tw, bool inverse)
{
    const int n = (int)x.size();
    Line y(n);
    int ns = 1;
    for (int m = n, R = 4; m > 1; ) {
        while (m % R) {
            R = R == 4 ? 2 : R == 2 ? 3 : R + 2;
            if (R * R > m) R = m;
        }
        m /= R;
        for (int pos = 0; pos < n; ++pos) {
            const int k = pos % ns, r = pos / ns % R, j = pos / (ns * R) * ns + k;
            const int step = k * (n / (ns * R)) + r * (n / R);
            c128 acc = x[j];
            for (int q = 1, e = 0; q < R; ++q) {
                e = (e + step) % n;
                acc = acc + mul(x[j + q * (n / R)], inverse ? conj(tw[e]) : tw[e]);
            }
            y[pos] = acc;
        }
        x.swap(y);
        ns *= R;
    }
}

static void exact(std::vector<cl> &x, const std::vector<cl> &w, size_t stride)
{
    const size_t n = x.size();
    if (n == 1) return;
    size_t p = 2;
    while (n % p) ++p;
    std::vector<std::vector<cl>> s(p, std::vector<cl>(n / p));
    for (size_t i = 0; i < n; ++i) s[i % p][i / p] = x[i];
    for (auto &v : s) exact(v, w, stride * p);
    for (size_t k = 0; k < n; ++k) {
        cl t = 0;
        for (size_t q = 0; q < p; ++q) t += s[q][k % (n / p)] * w[q * k % n * stride];
        x[k] = t;
    }
}

static ld rel(const Line &a, const std::vector<cl> &b)
{
    ld e = 0, r = 0;
    for (size_t i = 0; i < a.size(); ++i) {
        e += std::norm(cl(a[i].x, a[i].y) - b[i]);
        r += std::norm(b[i]);
    }
    return sqrtl(e / r);
}

static void swap_parts(Line &x)
{
    for (c128 &v : x) v = mk(v.y, v.x);
}

int main()
{
    int failures = 0, count = 0;
    ld once = 0, steps = 0;
    for (int n : {36, 96, 100, 144, 160, 216, 250, 300, 320, 360, 432, 500, 640, 720, 729, 750, 850,
                  864, 1000, 1250, 1331, 1500, 1800, 2187, 2401}) {
        MixPlan p;
        if (!mix_plan(n, n, &p)) return 1;
        Line tw(n), ev(n), kt(n), x(n);
        std::vector<cl> w(n), xl(n);
        unsigned s = 12345u + n;
        auto rnd = [&] {
            s = s * 1664525u + 1013904223u;
            return (s >> 8) / 8388608.0 - 1.0;
        };
        for (int m = 0; m < n; ++m) {
            const ld a = -2.0L * kPi * m / n;
            w[m] = cl(cosl(a), sinl(a));
            tw[m] = mk((double)cosl(a), (double)sinl(a));
            x[m].x = rnd();
            x[m].y = rnd();
            xl[m] = cl(x[m].x, x[m].y);
        }
        Line a = x, b = x;
        mixed(a, p.f, p.nf, tw);
        direct(b, tw, false);
        exact(xl, w, 1);
        once += logl(rel(a, xl) / rel(b, xl));
        // a packet, a barrier's and the kinetic phases (grid step 0.1, time
        // step 0.05, the middle stage of a fourth order step)
        const ld half = 0.05L * n;
        const double k0 = 1.5 + 0.5 * rnd(), at = 0.4 + 0.1 * rnd();
        for (int m = 0; m < n; ++m) {
            const ld q = -half + 0.1L * m, am = expl(-powl((q + half * at) / (0.14L * half), 2) / 2);
            x[m] = mk((double)(am * cosl(k0 * q)), (double)(am * sinl(k0 * q)));
            const cl f = std::polar(1.0L, -0.05L * 0.6756L * 0.7L * expl(-q * q / 1.4L));
            ev[m] = mk((double)f.real(), (double)f.imag());
            const ld k = (m > n / 2 ? n - m : m) * 2 * kPi / (0.1L * n);
            const cl g = std::polar(1.0L, -0.05L * 1.35L * k * k / 2);
            kt[m] = mk((double)g.real(), (double)g.imag());
            xl[m] = cl(x[m].x, x[m].y);
        }
        a = b = x;
        const double r = 1.0 / n;
        for (int t = 0; t < 60; ++t) {
            for (int i = 0; i < n; ++i) {
                a[i] = mul(a[i], ev[i]);
                b[i] = mul(b[i], ev[i]);
                xl[i] *= cl(ev[i].x, ev[i].y);
            }
            mixed(a, p.f, p.nf, tw);
            direct(b, tw, false);
            exact(xl, w, 1);
            for (int i = 0; i < n; ++i) {
                a[i] = mul(a[i], kt[i]);
                b[i] = mul(b[i], kt[i]);
                xl[i] = std::conj(xl[i] * cl(kt[i].x, kt[i].y));
            }
            swap_parts(a);
            mixed(a, p.f + kMixMaxPasses, p.nf, tw);
            swap_parts(a);
            direct(b, tw, true);
            exact(xl, w, 1);
            for (int i = 0; i < n; ++i) {
                a[i] = mix_scale(a[i], r, mix_recip_lo(n));
                b[i] = b[i] * r;
                xl[i] = std::conj(xl[i]) / (ld)n;
            }
        }
        const ld q = rel(a, xl) / rel(b, xl);
        steps += logl(q);
        ++count;
        if (!(q < 1.2L)) {
            std::printf("n=%d: after 60 steps %.2Lf times the error of direct sums\n", n, q);
            ++failures;
        }
    }
    once = expl(once / count);
    steps = expl(steps / count);
    std::printf("error beside direct sums: one transform %.3Lf, 60 steps %.3Lf\n", once, steps);
    if (!(once < 1) || !(steps < 1)) ++failures;
    if (!failures) std::printf("error growth ok\n");
    return failures != 0;
}
