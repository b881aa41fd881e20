// gf_fft_line.h — mixed-radix line transforms of the FFT passes, in
// registers with LDS exchanges between the radix passes.
//
// A line of length n is a product of at most kMaxPasses radices of
// {1..10, 12, 14, 15, 16}: two for most lengths up to 256, three up to 2048.
// Each pass gives a thread one butterfly: R elements read together, the
// R-point DFT in registers, R elements written (Stockham order: pass s of
// radix R over sub-transforms of size L, the product of the radices before
// it, reads elements j + r n/R, multiplies element r by w^(r k n/(L R)) with
// k = j mod L, and writes element q to (j div L) L R + k + q L, so natural
// order goes in and comes out).  The first pass reads its elements straight
// from global memory and the last writes straight to it, so a two-radix
// line crosses LDS once, behind one barrier, and all of a workgroup's global
// loads are in flight together.  The launches are bound by that one chain of
// memory round trip, butterflies and barriers, not by bandwidth: on a
// 100x84x30 grid (13 MB a pass) they take 6-12 us, against 11-15 us with
// radices of at most 7, every pass through LDS and a runtime integer
// division per element.
#pragma once

#include "gf_internal.h"

namespace gf {
namespace line {

__device__ __forceinline__ double2 mk(double a, double b) { return make_double2(a, b); }
__device__ __forceinline__ double2 add(double2 a, double2 b) { return mk(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 sub(double2 a, double2 b) { return mk(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 mul(double2 a, double2 b) {
    return mk(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a times the quarter turn of the transform's sign: -i forward, +i inverse
template <bool kInv>
__device__ __forceinline__ double2 quarter(double2 a) {
    return kInv ? mk(-a.y, a.x) : mk(a.y, -a.x);
}
template <bool kInv>
__device__ __forceinline__ double2 twiddle(double2 a, double2 w) {
    return mul(a, kInv ? mk(w.x, -w.y) : w);
}

// cos and sin of 2 pi k / R, rounded to double.
constexpr double kC5[5] = {1., 0.309016994374947424102, -0.809016994374947424102, -0.809016994374947424102,
                           0.309016994374947424102};
constexpr double kS5[5] = {0., 0.951056516295153572116, 0.587785252292473129169, -0.587785252292473129169,
                           -0.951056516295153572116};
constexpr double kC7[7] = {1., 0.623489801858733530525, -0.222520933956314404289, -0.900968867902419126236,
                           -0.900968867902419126236, -0.222520933956314404289, 0.623489801858733530525};
constexpr double kS7[7] = {0., 0.781831482468029808708, 0.974927912181823607018, 0.433883739117558120475,
                           -0.433883739117558120475, -0.974927912181823607018, -0.781831482468029808708};
constexpr double kC9[5] = {1., 0.766044443118978035202, 0.173648177666930348852, -0.5, -0.939692620785908384054};
constexpr double kS9[5] = {0., 0.642787609686539326323, 0.984807753012208059367, 0.866025403784438646764,
                           0.342020143325668733044};
constexpr double kHalf2 = 0.707106781186547524401;    // cos(pi/4)
constexpr double kC16 = 0.923879532511286756128, kS16 = 0.382683432365089771728;
constexpr double kSin60 = 0.866025403784438646764;

// exp(-2 pi i k / R) of the composite radices' inner twiddles
template <int R>
__host__ __device__ constexpr double2 inner(int k) {
    double c = 1., s = 0.;
    if (R == 8) {
        c = k == 0 ? 1. : k == 1 ? kHalf2 : k == 2 ? 0. : -kHalf2;
        s = k == 0 ? 0. : k == 2 ? 1. : kHalf2;
    } else if (R == 9) {
        c = kC9[k]; s = kS9[k];
    } else if (R == 16) {
        const double cs[10] = {1., kC16, kHalf2, kS16, 0., -kS16, -kHalf2, -kC16, -1., -kC16};
        const double sn[10] = {0., kS16, kHalf2, kC16, 1., kC16, kHalf2, kS16, 0., -kS16};
        c = cs[k]; s = sn[k];
    }
    return double2{c, -s};
}

template <int R, bool kInv>
struct Dft;

template <bool kInv>
struct Dft<1, kInv> {
    static __device__ __forceinline__ void run(double2 (&)[1]) {}
};
template <bool kInv>
struct Dft<2, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[2]) {
        const double2 a = v[0], b = v[1];
        v[0] = add(a, b);
        v[1] = sub(a, b);
    }
};
template <bool kInv>
struct Dft<3, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[3]) {
        const double2 s = add(v[1], v[2]), d = sub(v[1], v[2]);
        const double2 t = mk(v[0].x - 0.5 * s.x, v[0].y - 0.5 * s.y);
        const double2 q = quarter<kInv>(mk(kSin60 * d.x, kSin60 * d.y));
        v[0] = add(v[0], s);
        v[1] = add(t, q);
        v[2] = sub(t, q);
    }
};
template <bool kInv>
struct Dft<4, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[4]) {
        const double2 s0 = add(v[0], v[2]), d0 = sub(v[0], v[2]);
        const double2 s1 = add(v[1], v[3]), d1 = quarter<kInv>(sub(v[1], v[3]));
        v[0] = add(s0, s1);
        v[2] = sub(s0, s1);
        v[1] = add(d0, d1);
        v[3] = sub(d0, d1);
    }
};
// odd primes: elements r and R - r meet as a sum and a difference, so every
// product is by a real constant
template <int R, bool kInv>
__device__ __forceinline__ void dft_odd(double2 (&v)[R], const double (&C)[R], const double (&S)[R]) {
    constexpr int H = R / 2;
    double2 s[H], d[H], o[R];
#pragma unroll
    for (int m = 1; m <= H; m++) {
        s[m - 1] = add(v[m], v[R - m]);
        d[m - 1] = sub(v[m], v[R - m]);
    }
    o[0] = v[0];
#pragma unroll
    for (int m = 0; m < H; m++) o[0] = add(o[0], s[m]);
#pragma unroll
    for (int q = 1; q <= H; q++) {
        double2 A = v[0], B = mk(0., 0.);
#pragma unroll
        for (int m = 1; m <= H; m++) {
            const double c = C[(q * m) % R], w = S[(q * m) % R];
            A = mk(A.x + c * s[m - 1].x, A.y + c * s[m - 1].y);
            B = m == 1 ? mk(w * d[0].x, w * d[0].y) : mk(B.x + w * d[m - 1].x, B.y + w * d[m - 1].y);
        }
        B = quarter<kInv>(B);
        o[q] = add(A, B);
        o[R - q] = sub(A, B);
    }
#pragma unroll
    for (int q = 0; q < R; q++) v[q] = o[q];
}
template <bool kInv>
struct Dft<5, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[5]) { dft_odd<5, kInv>(v, kC5, kS5); }
};
template <bool kInv>
struct Dft<7, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[7]) { dft_odd<7, kInv>(v, kC7, kS7); }
};
// R = A B with inner twiddles: element B a + b, result ka + A kb
template <int A, int B, bool kInv>
__device__ __forceinline__ void dft_split(double2 (&v)[A * B]) {
    constexpr int R = A * B;
    double2 o[R];
#pragma unroll
    for (int b = 0; b < B; b++) {
        double2 t[A];
#pragma unroll
        for (int a = 0; a < A; a++) t[a] = v[B * a + b];
        Dft<A, kInv>::run(t);
#pragma unroll
        for (int k = 0; k < A; k++) {
            const int m = b * k;
            if (m == 0) o[B * k + b] = t[k];
            else if (4 * m == R) o[B * k + b] = quarter<kInv>(t[k]);
            else o[B * k + b] = twiddle<kInv>(t[k], inner<R>(m));
        }
    }
#pragma unroll
    for (int k = 0; k < A; k++) {
        double2 t[B];
#pragma unroll
        for (int b = 0; b < B; b++) t[b] = o[B * k + b];
        Dft<B, kInv>::run(t);
#pragma unroll
        for (int b = 0; b < B; b++) v[k + A * b] = t[b];
    }
}
// R = A B with A and B coprime (Good and Thomas): no inner twiddles; element
// (B a + A b) mod R, result the k with k = ka mod A, k = kb mod B
template <int A, int B, bool kInv>
__device__ __forceinline__ void dft_coprime(double2 (&v)[A * B]) {
    constexpr int R = A * B;
    double2 o[R];
#pragma unroll
    for (int b = 0; b < B; b++) {
        double2 t[A];
#pragma unroll
        for (int a = 0; a < A; a++) t[a] = v[(B * a + A * b) % R];
        Dft<A, kInv>::run(t);
#pragma unroll
        for (int k = 0; k < A; k++) o[B * k + b] = t[k];
    }
#pragma unroll
    for (int ka = 0; ka < A; ka++) {
        double2 t[B];
#pragma unroll
        for (int b = 0; b < B; b++) t[b] = o[B * ka + b];
        Dft<B, kInv>::run(t);
#pragma unroll
        for (int k = 0; k < R; k++)
            if (k % A == ka) v[k] = t[k % B];
    }
}
template <bool kInv>
struct Dft<6, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[6]) { dft_coprime<2, 3, kInv>(v); }
};
template <bool kInv>
struct Dft<8, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[8]) { dft_split<2, 4, kInv>(v); }
};
template <bool kInv>
struct Dft<9, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[9]) { dft_split<3, 3, kInv>(v); }
};
template <bool kInv>
struct Dft<10, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[10]) { dft_coprime<2, 5, kInv>(v); }
};
template <bool kInv>
struct Dft<12, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[12]) { dft_coprime<4, 3, kInv>(v); }
};
template <bool kInv>
struct Dft<14, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[14]) { dft_coprime<2, 7, kInv>(v); }
};
template <bool kInv>
struct Dft<15, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[15]) { dft_coprime<3, 5, kInv>(v); }
};
template <bool kInv>
struct Dft<16, kInv> {
    static __device__ __forceinline__ void run(double2 (&v)[16]) { dft_split<4, 4, kInv>(v); }
};

// x / d of a FastDiv (gf_internal.h).
__device__ __forceinline__ int div(const FastDiv& f, int x) {
    return f.d == 1u ? x : static_cast<int>(__umulhi(static_cast<uint32_t>(x), f.m));
}

// LDS slot of element i of a line: one spare slot after every 16 elements,
// so that the stride-R writes of a pass spread over the banks.
__device__ __forceinline__ int slot(int i) { return i + (i >> 4); }

// The thread's butterfly of a pass: line and j, or no butterfly.
struct Where {
    int line, j;
    bool on;
};
// lines vary fastest (2^loglines of them: consecutive threads take
// consecutive lines) or j does.
__device__ __forceinline__ Where where_line_fast(int per, int loglines) {
    const int t = threadIdx.x;
    return Where{t & ((1 << loglines) - 1), t >> loglines, (t >> loglines) < per};
}
__device__ __forceinline__ Where where_j_fast(const FastDiv& per, int lines) {
    const int t = threadIdx.x;
    const int l = div(per, t);
    return Where{l, t - l * static_cast<int>(per.d), l < lines};
}

// One butterfly: ld(element) reads each of its R inputs, cvt turns what it
// read into the complex value (after every read has been issued), then the
// DFT, and st(element, value) writes each output.
template <int R, bool kInv, bool kFirst, class Ld, class Cvt, class Sync, class St>
__device__ __forceinline__ void butterfly(const LinePlan& f, int s, Where w, const double2* tw, Ld ld, Cvt cvt,
                                          Sync sync, St st) {
    decltype(ld(0)) in[R];
    double2 v[R];
    const int per = static_cast<int>(f.per[s].d), L = static_cast<int>(f.L[s].d);
    if (w.on) {
#pragma unroll
        for (int r = 0; r < R; r++) in[r] = ld(w.j + r * per);
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = cvt(in[r], w.j + r * per);
    }
    sync();
    if (w.on) {
        int base = w.j * R, step = 1;
        if (!kFirst) {
            const int g = div(f.L[s], w.j), k = w.j - g * L;
            const int unit = k * f.unit[s];
#pragma unroll
            for (int r = 1; r < R; r++) v[r] = twiddle<kInv>(v[r], tw[r * unit]);
            base = g * L * R + k;
            step = L;
        }
        Dft<R, kInv>::run(v);
#pragma unroll
        for (int q = 0; q < R; q++) st(base + q * step, v[q]);
    }
}

// Pass s with the radix known at run time, at most kMaxR.  sync runs in
// every thread between the reads and the writes of the pass.
template <int kMaxR, bool kInv, bool kFirst, class Ld, class Cvt, class Sync, class St>
__device__ __forceinline__ void pass(const LinePlan& f, int s, Where w, const double2* tw, Ld ld, Cvt cvt, Sync sync,
                                     St st) {
#define GF_LINE_RADIX(R)                                                                             \
    case R:                                                                                          \
        if constexpr (R <= kMaxR) butterfly<R, kInv, kFirst>(f, s, w, tw, ld, cvt, sync, st);        \
        break
    switch (f.r[s]) {
        GF_LINE_RADIX(1);
        GF_LINE_RADIX(2);
        GF_LINE_RADIX(3);
        GF_LINE_RADIX(4);
        GF_LINE_RADIX(5);
        GF_LINE_RADIX(6);
        GF_LINE_RADIX(7);
        GF_LINE_RADIX(8);
        GF_LINE_RADIX(9);
        GF_LINE_RADIX(10);
        GF_LINE_RADIX(12);
        GF_LINE_RADIX(14);
        GF_LINE_RADIX(15);
        GF_LINE_RADIX(16);
    default: break;
    }
#undef GF_LINE_RADIX
}

struct Same {
    __device__ __forceinline__ double2 operator()(double2 v, int) const { return v; }
};

}  // namespace line
}  // namespace gf
