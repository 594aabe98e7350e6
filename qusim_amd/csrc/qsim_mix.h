// qsim_mix.h -- mixed-radix line transforms for lengths that are not a power
// of two (and for the short powers of two that have no fused kernel).
//
// mix_plan states which lengths run here.  It splits a length into 2..6
// radices of at most 15, with a pass of paired sums for each prime above 13
// (MixPlan); the kernels switch on the radix of each Stockham pass at run
// time, so one compiled kernel serves every such length.  A workgroup holds L lines (a power of two) in LDS, element m of
// line l at slot(m * L + l): lanes run over the lines first, so the
// exchanges of 4 or more lines touch whole 64-128 B runs whatever the radix,
// global loads of strided lines are coalesced, and the line index is a mask
// instead of a division.  Each pass loads its butterflies into registers,
// waits, and stores them back to the same LDS buffer: in place, which leaves
// room for twice the lines of a double-buffered exchange.
//
// Butterflies are computed in FP64 for both element types: FP32 VALU
// instructions issue at the FP64 rate here (packed FP32 is compiled out), so
// only the stored values round to FP32.
//
// The inverse transform is the forward one on values with real and imaginary
// parts swapped, so there is one set of butterflies.
#pragma once

#include <type_traits>

#include "qsim_common.h"

namespace qsim {

constexpr int kMixMaxPasses = 6;
constexpr int kMixMaxLen = 5120;
constexpr int kMixMaxThreads = 1024;
constexpr size_t kMixMaxLds = 160 * 1024;

struct MixPass {
    int R;           // radix
    int nb;          // butterflies of a line, n / R
    int ns;          // points combined by the passes before this one
    unsigned mag;    // ceil(2^32 / ns): j / ns = mulhi(j, mag) for j < 2^16
    int tws;         // twiddle step n / (ns R)
};

// A plan travels to the kernels by value (kernel arguments): a copy in device
// memory put one more dependent load in front of every sweep.
struct MixPlan {
    int n, nf;
    int tlen;                       // table entries that the passes use
    int prime;                      // has passes of a prime above 13
    MixPass f[2 * kMixMaxPasses];   // radices r0, r1, ... of the first transform;
                                    // from kMixMaxPasses on, in reverse order
};

// Butterflies of one thread per pass: 8 to 15 elements in registers, which
// leaves room for the factors of a pointwise stage beside them within the 128
// registers of a 1024-thread workgroup.
__host__ __device__ constexpr int mix_k(int R)
{
    return R == 1 ? 8 : R == 2 ? 4 : R == 3 ? 3 : R <= 7 ? 2 : 1;
}

// Slot of LDS element e: one element of padding per 8 (sh = 3), or per 16
// (sh = 4) where the longest lines leave no room for that.  The strided stores
// of the first pass then spread over the banks for even radices too (stride 4
// or 8 without padding: 4 and 8 lanes on one bank).
__host__ __device__ __forceinline__ int mix_slot(int e, int sh) { return e + (e >> sh); }

// ------------------------------------------------------------- butterflies
// A rounded constant repeats its rounding in every transform, and over the
// steps of an evolution that grows with their number, not with its root.
// Constants whose rounding showed (those of 3, 5, 8, 9 and 11 points) come as
// the double and the low part that the rounding took off; the low part goes
// into the addend of a product's fma, where the rounding that follows still
// moves by it, never onto a value alone.  7 and 13 points: MixPrime.

// cos and sin of 2 pi k / P, k = 1 .. (P-1)/2
template <int P>
struct MixC;
template <>
struct MixC<7> {
    static constexpr double c[3] = {0.62348980185873353053, -0.22252093395631440429,
                                    -0.90096886790241912624};
    static constexpr double s[3] = {0.78183148246802980871, 0.97492791218182360702,
                                    0.43388373911755812048};
    static constexpr bool LOW = false;
};
template <>
struct MixC<11> {
    static constexpr double c[5] = {0.84125353283118116886, 0.41541501300188642553,
                                    -0.14231483827328514044, -0.65486073394528506406,
                                    -0.95949297361449738988};
    static constexpr double s[5] = {0.54064081745559758211, 0.90963199535451837141,
                                    0.98982144188093273238, 0.75574957435425828377,
                                    0.28173255684142969771};
    static constexpr bool LOW = true;
    static constexpr double cl[5] = {-3.6647285149858677e-17, -9.5552123437671800e-18,
                                     3.1334476506295326e-18, 3.6553153571046389e-17,
                                     -2.1239679343678974e-17};
    static constexpr double sl[5] = {2.6677788920071333e-17, 4.1301477016464232e-17,
                                     4.8155296856458766e-17, 1.4869519672512073e-17,
                                     2.6676302681156600e-17};
};
template <>
struct MixC<13> {
    static constexpr double c[6] = {0.88545602565320989590, 0.56806474673115580251,
                                    0.12053668025532305335, -0.35460488704253562597,
                                    -0.74851074817110109863, -0.97094181742605202716};
    static constexpr double s[6] = {0.46472317204376854566, 0.82298386589365639458,
                                    0.99270887409805399280, 0.93501624268541482344,
                                    0.66312265824079520238, 0.23931566428755776714};
    static constexpr bool LOW = false;
};

__host__ __device__ __forceinline__ c128 mix_mi(c128 a) { return mk(a.y, -a.x); }  // -i a

// a + b c and a - b c, two roundings a component instead of the three of a
// product and a sum
__host__ __device__ __forceinline__ c128 mix_fma(c128 a, c128 b, c128 c)
{
    return mk(fma(-b.y, c.y, fma(b.x, c.x, a.x)), fma(b.y, c.x, fma(b.x, c.y, a.y)));
}
__host__ __device__ __forceinline__ c128 mix_fms(c128 a, c128 b, c128 c)
{
    return mk(fma(b.y, c.y, fma(-b.x, c.x, a.x)), fma(-b.y, c.x, fma(-b.x, c.y, a.y)));
}

// a w with w = h + l, l the low part
__host__ __device__ __forceinline__ c128 mix_mul(c128 a, c128 h, c128 l)
{
    return mix_fma(a * l, a, h);
}

// a / n by s = 1 / n, sl = mix_recip_lo(n): the rounding of 1 / n alone grew to
// 5e-15 over 60 steps of 243 or 850 points
__host__ __device__ __forceinline__ c128 mix_scale(c128 a, double s, double sl)
{
    return mk(fma(a.x, s, a.x * sl), fma(a.y, s, a.y * sl));
}
inline double mix_recip_lo(double n) { return fma(-(1.0 / n), n, 1.0) / n; }

// An R-point butterfly starts with sums and differences of pairs: pair(i, h)
// is element h (0, 1) of pair i.  rest() takes the sums in the first and the
// differences in the second places of the pairs and finishes the transform;
// elements in no pair enter as they are.
template <int R>
struct MixDft;

// An odd prime: X_m = x0 + sum_k (x_k + x_{P-k}) cos(2 pi k m / P)
//                        - i sum_k (x_k - x_{P-k}) sin(2 pi k m / P)
// The roundings of 7 and 13 points' constants left 60 steps of 343 to 3003
// points at 0.9 to 1.1 times the error of direct sums, so they take none of
// the low parts' instructions.
template <int P>
struct MixPrime {
    static constexpr int PAIRS = (P - 1) / 2;
    static __host__ __device__ constexpr int pair(int i, int h) { return h ? P - 1 - i : i + 1; }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        constexpr int H = PAIRS;
        c128 a[H], b[H], s0 = v[0];
        const c128 x0 = v[0];
#pragma unroll
        for (int k = 0; k < H; ++k) {
            a[k] = v[k + 1];
            b[k] = v[P - 1 - k];
            s0 = s0 + a[k];
        }
        v[0] = s0;
#pragma unroll
        for (int m = 1; m <= H; ++m) {
            constexpr bool LOW = MixC<P>::LOW;
            c128 e = LOW ? mk(0.0, 0.0) : x0, o = mk(0.0, 0.0);
            if constexpr (LOW) {
#pragma unroll
                for (int k = 1; k <= H; ++k) {
                    const int q = (k * m) % P, i = (q <= H ? q : P - q) - 1;
                    const double c = MixC<P>::cl[i];
                    const double s = q <= H ? MixC<P>::sl[i] : -MixC<P>::sl[i];
                    e = k == 1 ? mk(c * a[0].x, c * a[0].y)
                               : mk(fma(c, a[k - 1].x, e.x), fma(c, a[k - 1].y, e.y));
                    o = k == 1 ? mk(s * b[0].x, s * b[0].y)
                               : mk(fma(s, b[k - 1].x, o.x), fma(s, b[k - 1].y, o.y));
                }
            }
#pragma unroll
            for (int k = 1; k <= H; ++k) {
                const int q = (k * m) % P, i = (q <= H ? q : P - q) - 1;
                const double c = MixC<P>::c[i], s = q <= H ? MixC<P>::s[i] : -MixC<P>::s[i];
                e = mk(fma(c, a[k - 1].x, e.x), fma(c, a[k - 1].y, e.y));
                o = k == 1 && !LOW ? mk(s * b[0].x, s * b[0].y)
                                   : mk(fma(s, b[k - 1].x, o.x), fma(s, b[k - 1].y, o.y));
            }
            if constexpr (LOW) e = x0 + e;
            const c128 io = mix_mi(o);
            v[m] = e + io;
            v[P - m] = e - io;
        }
    }
};
// 3: the cosine is -1/2 exactly.
template <>
struct MixDft<3> {
    static constexpr int PAIRS = 1;
    static __host__ __device__ constexpr int pair(int, int h) { return 1 + h; }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        constexpr double s = 0.86602540378443864676, sl = 5.0175421109034514e-17;
        const c128 x0 = v[0], a = v[1], b = v[2];
        const c128 e = mk(fma(-0.5, a.x, x0.x), fma(-0.5, a.y, x0.y));
        const c128 o = mk(fma(s, b.y, sl * b.y), -fma(s, b.x, sl * b.x));   // -i o
        v[0] = x0 + a;
        v[1] = e + o;
        v[2] = e - o;
    }
};
// 5: the cosines' low parts are -q and q; the second sine's, a fifteenth of a
// unit, is left out.
template <>
struct MixDft<5> {
    static constexpr int PAIRS = 2;
    static __host__ __device__ constexpr int pair(int i, int h) { return h ? 4 - i : i + 1; }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
        constexpr double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
        constexpr double q = 2.7160576018412531e-17, l1 = 4.0934500900087295e-17;
        const c128 x0 = v[0], a1 = v[1], a2 = v[2], b1 = v[4], b2 = v[3];
        const c128 lo = q * (a2 - a1);
        const c128 e1 = mk(fma(c2, a2.x, x0.x) + fma(c1, a1.x, lo.x),
                           fma(c2, a2.y, x0.y) + fma(c1, a1.y, lo.y));
        const c128 e2 = mk(fma(c1, a2.x, x0.x) + fma(c2, a1.x, -lo.x),
                           fma(c1, a2.y, x0.y) + fma(c2, a1.y, -lo.y));
        const c128 o1 = mk(fma(s1, b1.y, fma(s2, b2.y, l1 * b1.y)),
                           -fma(s1, b1.x, fma(s2, b2.x, l1 * b1.x)));   // -i o
        const c128 o2 = mk(fma(s2, b1.y, -fma(s1, b2.y, l1 * b2.y)),
                           fma(-s2, b1.x, fma(s1, b2.x, l1 * b2.x)));
        v[0] = x0 + (a1 + a2);
        v[1] = e1 + o1;
        v[4] = e1 - o1;
        v[2] = e2 + o2;
        v[3] = e2 - o2;
    }
};
template <> struct MixDft<7> : MixPrime<7> {};
template <> struct MixDft<11> : MixPrime<11> {};
template <> struct MixDft<13> : MixPrime<13> {};

// A first or last pass that only loads or stores, beside a prime's pass.
template <>
struct MixDft<1> {
    static constexpr int PAIRS = 0;
    static __host__ __device__ constexpr int pair(int, int) { return 0; }
    static __host__ __device__ __forceinline__ void rest(c128 *) {}
};
template <>
struct MixDft<2> {
    static constexpr int PAIRS = 1;
    static __host__ __device__ constexpr int pair(int, int h) { return h; }
    static __host__ __device__ __forceinline__ void rest(c128 *) {}
};
template <>
struct MixDft<4> {
    static constexpr int PAIRS = 2;
    static __host__ __device__ constexpr int pair(int i, int h) { return i + 2 * h; }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        const c128 a = v[0], b = v[2], c = v[1], d = mix_mi(v[3]);
        v[0] = a + c;
        v[1] = b + d;
        v[2] = a - c;
        v[3] = b - d;
    }
};

template <int R>
__host__ __device__ __forceinline__ void mix_dft(c128 *v)
{
#pragma unroll
    for (int i = 0; i < MixDft<R>::PAIRS; ++i) {
        c128 &p = v[MixDft<R>::pair(i, 0)], &q = v[MixDft<R>::pair(i, 1)];
        const c128 a = p + q;
        q = p - q;
        p = a;
    }
    MixDft<R>::rest(v);
}

// R = A * B with a common factor: x[B a + b], X[k1 + A k2]; inner DFT_A over
// a, factor w_R^(b k1), DFT_B over b.
template <>
struct MixDft<8> {
    static constexpr int PAIRS = 4;
    static __host__ __device__ constexpr int pair(int i, int h) { return i + 4 * h; }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        auto mul = [](double x) {   // by sqrt(1/2)
            return fma(0.70710678118654752440, x, -4.8336466567264567e-17 * x);
        };
        c128 u[4] = {v[0], v[1], v[2], v[3]};
        c128 w[4] = {v[4], mk(mul(v[5].x + v[5].y), mul(v[5].y - v[5].x)), mix_mi(v[6]),
                     mk(mul(v[7].y - v[7].x), -mul(v[7].x + v[7].y))};
        mix_dft<4>(u);
        mix_dft<4>(w);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            v[2 * q] = u[q];
            v[2 * q + 1] = w[q];
        }
    }
};
template <>
struct MixDft<9> {
    static constexpr int PAIRS = 3;
    static __host__ __device__ constexpr int pair(int i, int h) { return 3 + i + 3 * h; }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        // w_9^1, w_9^2, w_9^4 and their low parts
        constexpr c128 w1 = {0.76604444311897803520, -0.64278760968653932632},
                       w2 = {0.17364817766693034885, -0.98480775301220805937},
                       w4 = {-0.93969262078590838405, -0.34202014332566873304},
                       l1 = {2.1750711742081045e-17, 3.6596079007909491e-17},
                       l2 = {-1.0090493350843633e-17, -3.9051088757992981e-17},
                       l4 = {4.3850932840020416e-17, -2.0136016534644645e-17};
        c128 t[3][3];
#pragma unroll
        for (int b = 0; b < 3; ++b) {
#pragma unroll
            for (int a = 0; a < 3; ++a) t[b][a] = v[3 * a + b];
            MixDft<3>::rest(t[b]);
        }
        t[1][1] = mix_mul(t[1][1], w1, l1);
        t[1][2] = mix_mul(t[1][2], w2, l2);
        t[2][1] = mix_mul(t[2][1], w2, l2);
        t[2][2] = mix_mul(t[2][2], w4, l4);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            c128 u[3] = {t[0][k], t[1][k], t[2][k]};
            mix_dft<3>(u);
#pragma unroll
            for (int q = 0; q < 3; ++q) v[k + 3 * q] = u[q];
        }
    }
};

// R = 2 B, B odd (Good and Thomas): x[(B a + 2 b) mod R],
// X[(B k1 + 2 (2^-1 mod B) k2) mod R], no factors between.
template <int B>
struct MixTwice {
    static constexpr int R = 2 * B, PAIRS = B;
    static __host__ __device__ constexpr int pair(int i, int h) { return (B * h + 2 * i) % R; }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        constexpr int EB = 2 * ((B + 1) / 2);
        c128 t[2][B];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
#pragma unroll
            for (int b = 0; b < B; ++b) t[k][b] = v[(B * k + 2 * b) % R];
            mix_dft<B>(t[k]);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int q = 0; q < B; ++q) v[(B * k + EB * q) % R] = t[k][q];
    }
};
template <> struct MixDft<6> : MixTwice<3> {};
template <> struct MixDft<10> : MixTwice<5> {};
template <> struct MixDft<14> : MixTwice<7> {};

// Likewise 12 = 4 * 3: x[(3 a + 4 b) mod 12], X[(9 k1 + 4 k2) mod 12]; the
// pairs are the first half of the 4-point transforms over a.
template <>
struct MixDft<12> {
    static constexpr int PAIRS = 6;
    static __host__ __device__ constexpr int at(int a, int b) { return (3 * a + 4 * b) % 12; }
    static __host__ __device__ constexpr int pair(int i, int h) { return at(i % 2 + 2 * h, i / 2); }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        c128 t[4][3];
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            c128 u[4] = {v[at(0, b)], v[at(1, b)], v[at(2, b)], v[at(3, b)]};
            MixDft<4>::rest(u);
#pragma unroll
            for (int k = 0; k < 4; ++k) t[k][b] = u[k];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            mix_dft<3>(t[k]);
#pragma unroll
            for (int q = 0; q < 3; ++q) v[(9 * k + 4 * q) % 12] = t[k][q];
        }
    }
};

// and 15 = 3 * 5: x[(5 a + 3 b) mod 15], X[(10 k1 + 6 k2) mod 15]
template <>
struct MixDft<15> {
    static constexpr int PAIRS = 5;
    static __host__ __device__ constexpr int at(int a, int b) { return (5 * a + 3 * b) % 15; }
    static __host__ __device__ constexpr int pair(int i, int h) { return at(1 + h, i); }
    static __host__ __device__ __forceinline__ void rest(c128 *v)
    {
        c128 t[3][5];
#pragma unroll
        for (int b = 0; b < 5; ++b) {
            c128 u[3] = {v[at(0, b)], v[at(1, b)], v[at(2, b)]};
            MixDft<3>::rest(u);
#pragma unroll
            for (int k = 0; k < 3; ++k) t[k][b] = u[k];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            mix_dft<5>(t[k]);
#pragma unroll
            for (int q = 0; q < 5; ++q) v[(10 * k + 6 * q) % 15] = t[k][q];
        }
    }
};

// Twiddles of one butterfly, w^r for r < R, each a rounded table entry read
// where it is used (the table stays in LDS).  With w^4 + q and w^8 + q as
// products of two entries 1000 points cost 315 us instead of 333 (O4, 20 steps),
// but after 60 transform pairs (on the CPU, 51 lengths, the same inputs) the
// error was 1.36 times that of direct sums in the mean instead of 1.19 (all
// with the butterflies' constants still rounded once).
template <int R>
struct MixTw {
    const c128 *t;
    int i;
    // tw: the table in LDS
    __host__ __device__ __forceinline__ void load(const c128 *tw, int idx)
    {
        t = tw;
        i = idx;
    }
    __host__ __device__ __forceinline__ c128 get(int r) const { return t[r * i]; }
    // the butterfly of the twiddled inputs, the products inside the sums and
    // differences of the pairs (as many operations as apart, fewer roundings:
    // the error is that of a direct sum with table factors)
    __host__ __device__ __forceinline__ void dft(c128 *v) const
    {
        bool done[R] = {};
        done[0] = true;
#pragma unroll
        for (int i = 0; i < MixDft<R>::PAIRS; ++i) {
            const int p = MixDft<R>::pair(i, 0), q = MixDft<R>::pair(i, 1);
            const c128 t = p == 0 ? v[0] : v[p] * get(p), y = v[q], w = get(q);
            v[p] = mix_fma(t, y, w);
            v[q] = mix_fms(t, y, w);
            done[p] = done[q] = true;
        }
#pragma unroll
        for (int r = 1; r < R; ++r)
            if (!done[r]) v[r] = v[r] * get(r);
        MixDft<R>::rest(v);
    }
};

// ----------------------------------------------------------------- passes
// One workgroup's lines: L = 1 << logl lines of plan length n in `lds`; the
// twiddle table's first tlen entries in `tw` (LDS too).
template <typename T>
struct MixWg {
    cx<T> *lds, *alt;   // read by the next pass; written by it (lds: in place)
    const c128 *tw;
    int tid, nt, logl, sh;
};

__host__ __device__ __forceinline__ unsigned mix_mulhi(unsigned a, unsigned b)
{
    return (unsigned)(((unsigned long long)a * b) >> 32);
}
// j % ns of a pass
__host__ __device__ __forceinline__ int mix_mod(const MixPass &p, int j)
{
    return p.ns == 1 ? 0 : j - (int)mix_mulhi((unsigned)j, p.mag) * p.ns;
}

__device__ __forceinline__ c128 mix_swap(c128 a) { return mk(a.y, a.x); }

template <typename T>
__device__ __forceinline__ c128 mix_ld(const MixWg<T> &w, int l, int m)
{
    return cvt<double>(w.lds[mix_slot((m << w.logl) + l, w.sh)]);
}
template <typename T>
__device__ __forceinline__ void mix_st(const MixWg<T> &w, int l, int m, c128 v)
{
    w.alt[mix_slot((m << w.logl) + l, w.sh)] = cvt<T>(v);
}

// Launch shape as a kernel argument (blockDim and gridDim are read from hidden
// arguments, two dependent loads at the start of every kernel).
struct MixDims {
    int nt, logl, sh;  // threads, log2 of the lines per workgroup, mix_slot's sh
    int alt;           // elements between the two LDS buffers (0: in place)
    unsigned blocks;
};

// The workgroup's view of its dynamic LDS: the twiddles, then the lines.  The
// table is copied straight to LDS (no registers); the loads are issued before
// the first pass reads its lines and are waited for before its barrier, so
// every later pass finds its twiddles at LDS latency.  (Read from L2 in every
// pass, they made a 750 x 600 sweep wait for 80% of its wave cycles.)
template <typename T>
__device__ __forceinline__ MixWg<T> mix_begin(unsigned char *smem, const MixPlan &p, MixDims d,
                                              const c128 *tw)
{
    c128 *t = reinterpret_cast<c128 *>(smem);
    const int lane = threadIdx.x & 63;
    for (int b = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63); b < p.tlen; b += d.nt)
        if (b + lane < p.tlen)
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void *)(tw + b + lane),
                (__attribute__((address_space(3))) void *)(t + b), 16, 0, 0);
    cx<T> *lds = reinterpret_cast<cx<T> *>(t + p.tlen);
    return MixWg<T>{lds, lds + d.alt, t, (int)threadIdx.x, d.nt, d.logl, d.sh};
}

// vmcnt(0): the table's loads are done (before a barrier)
__device__ __forceinline__ void mix_wait_table() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// The kinds of pass.  FIRST reads `in` and has no twiddles; HEAD is a first
// pass on lines that are in LDS already; LAST writes `out`; TURN is the last pass of one transform, the pointwise stage `mid`
// and the first pass of the next transform (whose first radix is this one's
// last, so its inputs are already in the right registers).
enum { MIX_FIRST = 0, MIX_MID = 1, MIX_TURN = 2, MIX_LAST = 3, MIX_HEAD = 4 };

// pre(l, m): the factor of `mid` and `out` at element m, loaded at the top of
// the pass so that it lands while the butterflies run; fn(l, m, v, factor).
struct MixNoPre {
    __device__ __forceinline__ c128 operator()(int, int) const { return mk(0.0, 0.0); }
};

template <int KIND, int R, int PREMAX, typename T, typename Pre, typename F>
__device__ __forceinline__ void mix_pass_r(const MixWg<T> &w, const MixPass &p, Pre pre, F fn)
{
    constexpr int K = mix_k(R);
    constexpr bool HAS = !std::is_same<Pre, MixNoPre>::value;
    // the first butterfly's factors, as far as the registers go; the others
    // are loaded where they are used
    constexpr bool PRE = HAS && R <= PREMAX && (PREMAX > 9 || K * R <= 9);
    const int total = p.nb << w.logl, lm = (1 << w.logl) - 1;
    c128 v[K][R], f[PRE ? R : 1];
    MixTw<R> tw;
#pragma unroll
    for (int u = 0; u < K; ++u) {
        const int q = w.tid + u * w.nt;
        if (q < total) {
            const int l = q & lm, j = q >> w.logl;
            const int k = KIND == MIX_LAST ? mix_mod(p, j) : 0, base = (j - k) * R + k;
            if (PRE && u == 0) {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    f[PRE ? r : 0] = KIND == MIX_LAST ? pre(l, base + r * p.ns) : pre(l, j + r * p.nb);
            }
            if constexpr (KIND != MIX_FIRST && KIND != MIX_HEAD)
                if (u == 0) tw.load(w.tw, mix_mod(p, j) * p.tws);
#pragma unroll
            for (int r = 0; r < R; ++r)
                v[u][r] = KIND == MIX_FIRST ? fn(l, j + r * p.nb, mk(0.0, 0.0), mk(0.0, 0.0))
                                            : mix_ld(w, l, j + r * p.nb);
        }
    }
    // in place: everything read before anything is overwritten
    if constexpr (KIND == MIX_MID || KIND == MIX_TURN || KIND == MIX_HEAD)
        if (w.lds == w.alt) __syncthreads();
#pragma unroll
    for (int u = 0; u < K; ++u) {
        const int q = w.tid + u * w.nt;
        if (q < total) {
            const int l = q & lm, j = q >> w.logl;
            const int k = KIND == MIX_TURN ? j : mix_mod(p, j), base = (j - k) * R + k;
            if constexpr (KIND != MIX_FIRST && KIND != MIX_HEAD) {
                if (u > 0) tw.load(w.tw, k * p.tws);
                tw.dft(v[u]);
            } else {
                mix_dft<R>(v[u]);
            }
            if constexpr (KIND == MIX_TURN) {
                // outputs at j + r nb: the inputs of the next first pass
#pragma unroll
                for (int r = 0; r < R; ++r)
                    v[u][r] = fn(l, j + r * p.nb, v[u][r],
                                 PRE && u == 0 ? f[PRE ? r : 0] : pre(l, j + r * p.nb));
                mix_dft<R>(v[u]);
#pragma unroll
                for (int r = 0; r < R; ++r) mix_st(w, l, j * R + r, v[u][r]);
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if constexpr (KIND == MIX_LAST)
                        (void)fn(l, base + r * p.ns, v[u][r],
                                 PRE && u == 0 ? f[PRE ? r : 0] : pre(l, base + r * p.ns));
                    else mix_st(w, l, base + r * p.ns, v[u][r]);
                }
            }
        }
    }
    if constexpr (KIND == MIX_FIRST) mix_wait_table();
    if constexpr (KIND != MIX_LAST) __syncthreads();
}

// A pass of a prime P above 13.  First the twiddled inputs' pairs (k, P - k),
// in place: a_k = x_k + x_{P-k}, b_k = x_k - x_{P-k}; then the outputs m and
// P - m of butterfly j, X = x_0 + sum_k a_k cos(2 pi k m / P) -+ i sum_k b_k
// sin(2 pi k m / P).  at(e): element e of the line.  Against one sum of P
// terms per output it takes half the LDS reads, and its error is smaller.
template <typename At>
__host__ __device__ __forceinline__ void mix_prime_pair(const MixPass &p, const c128 *tw, int j,
                                                        int k, At at)
{
    const int e = k * mix_mod(p, j) * p.tws, f = (p.R - k) * mix_mod(p, j) * p.tws;
    const c128 x = at.get(j + k * p.nb) * tw[e], y = at.get(j + (p.R - k) * p.nb), w = tw[f];
    at.set(j + k * p.nb, mix_fma(x, y, w));
    at.set(j + (p.R - k) * p.nb, mix_fms(x, y, w));
}
// Outputs m, m + dm, ... of one butterfly (M of them, those up to (P - 1) / 2):
// a_k and b_k are read once for all.
template <int M, typename At, typename Out>
__host__ __device__ __forceinline__ void mix_prime_out(const MixPass &p, const c128 *tw, int j,
                                                       int m, int dm, At at, Out out)
{
    const int P = p.R, H = (P - 1) / 2, k0 = mix_mod(p, j), base = (j - k0) * P + k0;
    c128 e[M], o[M];
    int q[M], mi[M];
    const c128 x0 = at.get(j);
#pragma unroll
    for (int i = 0; i < M; ++i) {
        mi[i] = m + i * dm <= H ? m + i * dm : m;   // past the last: the first again
        q[i] = 0;
        e[i] = x0;
        o[i] = mk(0.0, 0.0);
    }
    for (int k = 1; 2 * k < P; ++k) {
        const c128 a = at.get(j + k * p.nb), b = at.get(j + (P - k) * p.nb);
#pragma unroll
        for (int i = 0; i < M; ++i) {
            q[i] += mi[i];
            if (q[i] >= P) q[i] -= P;
            const c128 w = tw[q[i] * p.nb];
            e[i] = mk(fma(w.x, a.x, e[i].x), fma(w.x, a.y, e[i].y));
            o[i] = mk(fma(-w.y, b.y, o[i].x), fma(w.y, b.x, o[i].y));   // i sum w.y b
        }
    }
#pragma unroll
    for (int i = 0; i < M; ++i)
        if (m + i * dm <= H) {
            out(base + mi[i] * p.ns, e[i] + o[i]);
            if (mi[i] > 0) out(base + (P - mi[i]) * p.ns, e[i] - o[i]);
        }
}

template <typename T>
__device__ __forceinline__ void mix_prime(const MixWg<T> &w, const MixPass &p)
{
    struct At {
        const MixWg<T> &w;
        int l;
        __device__ __forceinline__ c128 get(int e) const { return mix_ld(w, l, e); }
        __device__ __forceinline__ void set(int e, c128 v) const
        {
            w.lds[mix_slot((e << w.logl) + l, w.sh)] = cvt<T>(v);
        }
    };
    const int lm = (1 << w.logl) - 1, H = (p.R - 1) / 2;
    const unsigned mag = p.nb == 1 ? 0u : 0xffffffffu / (unsigned)p.nb + 1u;
    const int pairs = (p.nb * H) << w.logl;
    for (int q = w.tid; q < pairs; q += w.nt) {
        const int t = q >> w.logl, k = p.nb == 1 ? t : (int)mix_mulhi((unsigned)t, mag);
        mix_prime_pair(p, w.tw, t - k * p.nb, k + 1, At{w, q & lm});
    }
    __syncthreads();
    auto outputs = [&](auto mc) {
        constexpr int M = decltype(mc)::value;
        const int dm = (H + M) / M, outs = (p.nb * dm) << w.logl;
        for (int q = w.tid; q < outs; q += w.nt) {
            const int t = q >> w.logl, m = p.nb == 1 ? t : (int)mix_mulhi((unsigned)t, mag);
            mix_prime_out<M>(p, w.tw, t - m * p.nb, m, dm, At{w, q & lm},
                             [&](int e, c128 v) { mix_st(w, q & lm, e, v); });
        }
    };
    // as many outputs per thread as one round of the threads needs: alone an
    // output is bound by LDS reads, three for four FMAs (1D step of 2003 points
    // 438 us with 1, 282 with 4), but idle threads cost more (997 points 112 us
    // with 1, 145 with 4)
    const int all = (p.nb * (H + 1)) << w.logl;
    if (all <= w.nt) outputs(std::integral_constant<int, 1>());
    else if (all <= 2 * w.nt) outputs(std::integral_constant<int, 2>());
    else outputs(std::integral_constant<int, 4>());
    __syncthreads();
}

template <int KIND, int PREMAX = 9, typename T, typename Pre, typename F>
__device__ __forceinline__ void mix_pass(MixWg<T> &w, const MixPass &pass, Pre pre, F fn)
{
    // an opaque copy of the thread index: in a loop over steps the compiler
    // would otherwise hoist the addresses of all the radices out of it
    MixWg<T> wq = w;
    asm volatile("" : "+v"(wq.tid));
    // the whole pass description in one scalar load, not one per use
    const MixPass p = pass;
    asm volatile("" ::"s"(p.R), "s"(p.nb), "s"(p.ns), "s"(p.mag), "s"(p.tws));
    switch (p.R) {
#define QSIM_MIX_R(R_) \
    case R_: mix_pass_r<KIND, R_, PREMAX>(wq, p, pre, fn); break;
        QSIM_MIX_R(1) QSIM_MIX_R(2) QSIM_MIX_R(3) QSIM_MIX_R(4) QSIM_MIX_R(5) QSIM_MIX_R(6) QSIM_MIX_R(7)
        QSIM_MIX_R(8) QSIM_MIX_R(9) QSIM_MIX_R(10) QSIM_MIX_R(11) QSIM_MIX_R(12) QSIM_MIX_R(13)
        QSIM_MIX_R(14) QSIM_MIX_R(15)
#undef QSIM_MIX_R
        default:
            if constexpr (KIND == MIX_MID) mix_prime(wq, p);
            break;
    }
    if constexpr (KIND != MIX_LAST) {
        w.lds = wq.alt;
        w.alt = wq.lds;
    }
}

// passes 1 .. nf - 2 of a transform (rev: in the reverse radix order)
template <typename T>
__device__ __forceinline__ void mix_inner(MixWg<T> &w, const MixPlan &p, bool rev)
{
    const int o = rev ? kMixMaxPasses : 0;
    for (int i = 1; i < p.nf - 1; ++i)
        mix_pass<MIX_MID>(w, p.f[o + i], MixNoPre(), [](int, int, c128 v, c128) { return v; });
}
__host__ __device__ __forceinline__ const MixPass &mix_last(const MixPlan &p, bool rev)
{
    return p.f[(rev ? kMixMaxPasses : 0) + p.nf - 1];
}

// One transform: in(l, m, -, -) -> values, out(l, m, v, pre(l, m)).
template <typename T, typename In, typename Pre, typename Out>
__device__ __forceinline__ void mix_one(MixWg<T> &w, const MixPlan &p, In in, Pre pre,
                                        Out out)
{
    mix_pass<MIX_FIRST>(w, p.f[0], MixNoPre(), in);
    mix_inner(w, p, false);
    mix_pass<MIX_LAST>(w, mix_last(p, false), pre, out);
}

// Two transforms with a pointwise stage between them.
template <typename T, typename In, typename Pre, typename Mid, typename Out>
__device__ __forceinline__ void mix_two(MixWg<T> &w, const MixPlan &p, In in, Pre pre,
                                        Mid mid, Out out)
{
    mix_pass<MIX_FIRST>(w, p.f[0], MixNoPre(), in);
    mix_inner(w, p, false);
    mix_pass<MIX_TURN>(w, mix_last(p, false), pre, mid);
    mix_inner(w, p, true);
    mix_pass<MIX_LAST>(w, mix_last(p, true), MixNoPre(), out);
}

// ------------------------------------------------------------ host planning
// Cycles of one pass when a CU holds `work` line elements at a time: a fixed
// part (LDS round trip, barriers, the scalar set-up of the pass) and the FP64
// instructions of its butterflies, 4 cycles each on one of 4 SIMDs.  The fixed
// part is fitted: 300, 700 and 1800 cycles make 4, 4 and 3 passes of a
// 1000-point line held alone (5.3, 5.3 and 5.7 us a step), 3, 2 and 2 of 360
// points (4.2, 3.8 and 3.8), and differ by less than 5% on grids (timed without
// the low parts; 1000 and 360 points take 6.1 and 4.6 us with them, of which the
// host's call is a part).
inline double mix_cost(int R, double work)
{
    // butterfly, twiddles and index arithmetic; of the low parts' instructions
    // only those of 9, 11 and 15 points are in (1920 x 1920 646 -> 603 us for 5
    // steps, 120^3 Born 582 -> 532, 972 points 443 -> 373, the rest within 1%):
    // with all, plans have more and smaller radices, at 900 x 900 177 us instead
    // of 163, and one transform is 1.2% further off in the mean
    const int instr = R == 2 ? 40 : R == 3 ? 60 : R == 4 ? 64 : R == 5 ? 96 : R == 6 ? 112
                      : R == 7 ? 146 : R == 8 ? 148 : R == 9 ? 240 : R == 10 ? 212
                      : R == 11 ? 384 : R == 12 ? 240 : R == 13 ? 348 : R == 14 ? 320 : 386;
    const double waves = work / (256.0 * R);
    return 700 + 4 * instr * (waves > 1 ? waves : 1);
}

// Splits n into 2..kMixMaxPasses radices of the least cost, largest first.
inline void mix_split(int n, int maxr, int depth, double work, double cost, int *cur, int *best,
                      int *best_nf, double *best_cost)
{
    if (n == 1) {
        if (depth >= 2 && cost < *best_cost) {
            *best_nf = depth;
            *best_cost = cost;
            for (int i = 0; i < depth; ++i) best[i] = cur[i];
        }
        return;
    }
    if (depth == kMixMaxPasses) return;
    for (int r = maxr; r >= 2; --r)
        if (n % r == 0) {
            cur[depth] = r;
            mix_split(n / r, r, depth + 1, work, cost + mix_cost(r, work), cur, best, best_nf,
                      best_cost);
        }
}

// The lengths of mixed-radix lines: composite numbers with prime factors of at
// most 13 from 4 to kMixMaxLen, and numbers with a larger prime factor, primes
// included, while the twiddles and two lines fit 160 KiB (mix_fits: every one
// up to 3150).  Not among them: 1 to 3, the primes 5 to 13, and from 3151 on
// most lengths with a prime factor above 13.  false for those, and *out is an
// empty plan (n = 0), which callers keep as "no mixed-radix line here".  `work`:
// line elements that a CU holds at a time.
bool mix_fits(const MixPlan &p);
inline bool mix_plan(size_t n, double work, MixPlan *out)
{
    *out = MixPlan{};
    MixPlan plan{}, *p = &plan;
    if (n < 4 || n > (size_t)kMixMaxLen) return false;
    int primes[kMixMaxPasses], np = 0, s = (int)n;
    for (int q = 17; q <= s; q += 2)
        while (s % q == 0) {   // q is prime or s has lost its factors
            bool is_prime = true;
            for (int d = 3; d * d <= q; d += 2) is_prime = is_prime && q % d;
            if (!is_prime) break;
            if (np == kMixMaxPasses - 2) return false;
            primes[np++] = q;
            s /= q;
        }
    int cur[kMixMaxPasses], best[kMixMaxPasses], nf = 0;
    double cost = 1e300;
    if (s > 1) mix_split(s, 15, 0, work, 0, cur, best, &nf, &cost);
    if (np > 0) {
        // the primes in the middle, between radices that may be 1
        if (nf == 0 && s <= 15) {
            best[0] = s;
            best[1] = 1;
            nf = 2;
        }
        if (nf == 0 || nf + np > kMixMaxPasses) return false;
        for (int i = nf - 1; i >= 1; --i) best[i + np] = best[i];
        for (int i = 0; i < np; ++i) best[1 + i] = primes[i];
        nf += np;
    }
    if (nf == 0) return false;
    p->prime = np > 0;
    p->n = (int)n;
    p->nf = nf;
    p->tlen = 0;
    for (int dir = 0; dir < 2; ++dir) {
        MixPass *f = p->f + (dir ? kMixMaxPasses : 0);
        int ns = 1;
        for (int i = 0; i < nf; ++i) {
            const int R = best[dir ? nf - 1 - i : i];
            f[i].R = R;
            f[i].nb = (int)n / R;
            f[i].ns = ns;
            f[i].mag = ns == 1 ? 0u : (unsigned)((0x100000000ull + ns - 1) / ns);
            f[i].tws = (int)n / (ns * R);
            int top = (R - 1) * (ns - 1) * f[i].tws + 1;
            if (R > 15 && (R - 1) * f[i].nb >= top) top = (R - 1) * f[i].nb + 1;
            if (top > p->tlen) p->tlen = top;
            ns *= R;
        }
    }
    if (!mix_fits(*p)) return false;
    *out = plan;
    return true;
}

// Elements of `nlines` lines of n points that one of 256 CUs holds at a time:
// at most two workgroups' lines.
inline double mix_work(size_t n, size_t nlines)
{
    const double w = (double)n * (double)nlines / 256;
    return w < 8192 ? w : 8192;
}

// Launch shape of a sweep and its LDS bytes.
struct MixShape {
    MixDims d;
    size_t lds;
};

// threads for `L` lines: one butterfly per thread in every pass, as far as
// the workgroup's limit goes; 0 when some pass would need more per thread
// than mix_k allows
inline int mix_threads(const MixPlan &p, int L)
{
    int nt = 64;
    for (int i = 0; i < p.nf; ++i) {
        const int R = p.f[i].R, total = p.f[i].nb * L;
        if (R > 15) {   // its outputs are a loop
            int t = (p.f[i].nb * (R + 1) / 2 * L + 63) / 64 * 64;
            if (t > 512) t = 512;
            if (t > nt) nt = t;
            continue;
        }
        const int per = total <= 512 && R > 1 ? 1 : mix_k(R);
        int t = ((total + per - 1) / per + 63) / 64 * 64;
        if (t > kMixMaxThreads) return 0;
        if (t > nt) nt = t;
    }
    return nt;
}

// Launch shape of L = 1 << lg lines per workgroup, with two LDS buffers (one
// barrier per pass instead of two) where they fit in `pair` bytes; nt = 0 when
// it does not fit a workgroup.
inline MixShape mix_shape_of(const MixPlan &p, int lg, size_t nlines, size_t elem_bytes,
                             size_t pair)
{
    const size_t n = (size_t)p.n << lg, tab = p.tlen * sizeof(c128);
    MixShape s{MixDims{mix_threads(p, 1 << lg), lg, 3, 0,
                       (unsigned)((nlines + ((size_t)1 << lg) - 1) >> lg)}, 0};
    size_t elems = n + (n >> 3);
    if (tab + elems * elem_bytes > kMixMaxLds) {
        s.d.sh = 4;
        elems = n + (n >> 4);
    }
    s.lds = tab + elems * elem_bytes;
    if (s.lds > kMixMaxLds) s.d.nt = 0;
    // a prime's pass does not run in place
    if (p.prime) {
        pair = kMixMaxLds;
        if (s.lds + elems * elem_bytes > pair) s.d.nt = 0;
    }
    if (s.lds + elems * elem_bytes <= pair) {
        s.d.alt = (int)elems;
        s.lds += elems * elem_bytes;
    }
    return s;
}

inline bool mix_fits(const MixPlan &p) { return mix_shape_of(p, 0, 1, sizeof(c128), 0).d.nt > 0; }

inline MixShape mix_shape(const MixPlan &p, size_t nlines, size_t elem_bytes, bool strided)
{
    // strided lines come in tiles of 64 B of adjacent lines where those fit a
    // workgroup (600 x 750 with tiles of 64 and 128 B: 27.1 and 29.8 us a step,
    // 1000 x 1000 36.9 and 40.1; 32 B: 34.4 and 45.1), other tiles in half the
    // LDS, so that two workgroups share a CU
    const int want = strided ? 64 / (int)elem_bytes : 1;
    int best = 0;
    for (int lg = 1; lg <= 6; ++lg) {
        const int L = 1 << lg;
        const MixShape t = mix_shape_of(p, lg, nlines, elem_bytes, 0);
        if (t.d.nt == 0 || (L > want && t.lds > kMixMaxLds / 2)) break;
        // a workgroup for each of 256 CUs comes before wider tiles
        if (L > want && (nlines + L - 1) / L < 256) break;
        if (L * (int)elem_bytes > 128 && p.n * L > 2048) break;
        best = lg;
    }
    const size_t per_cu = (((nlines + ((size_t)1 << best) - 1) >> best) + 255) / 256;
    return mix_shape_of(p, best, nlines, elem_bytes, kMixMaxLds / (per_cu < 4 ? per_cu : 4));
}

}  // namespace qsim
