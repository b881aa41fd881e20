// gf_fft_any.hip — FP64 magnetostatic and electrostatic FFT passes for
// grids whose sizes are not all powers of two.
//
// The reference plans cufftPlan3d(nx, ny, nz) for any grid
// (magnetic_initialize.cpp:114-115, ferroelectric_initialize.cpp:351-352).
// These kernels are the five passes of gf_fft.hip (same layouts, same
// tensor product) with the mixed-radix line transforms of gf_fft_line.h:
// lengths whose prime factors are 2, 3, 5 and 7.  A workgroup takes as many
// lines as keep its threads to one butterfly each; the y passes give
// consecutive threads consecutive x on the side of the [kz][y][x] buffer and
// consecutive y on the other, so both global sides run along memory.  The z
// passes transform two real columns as one complex line.
#include <algorithm>

#include "gf_fft_line.h"

namespace gf {

namespace {

using line::pass;
using line::slot;
using line::Where;

constexpr int kMaxThreads = 1024;

__device__ __forceinline__ void load_table(double2* dst, const double2* src, int n) {
    for (int t = threadIdx.x; t < n; t += blockDim.x) dst[t] = src[t];
}

// Element i of an array whose base is uniform over the workgroup, through a
// 32-bit byte offset: the base stays in scalar registers (a workgroup's lines
// span less than 4 GiB of a component).
template <class T>
__device__ __forceinline__ T load_at(const T* base, uint32_t i) {
    typedef const __attribute__((address_space(1))) char* Bytes;
    typedef const __attribute__((address_space(1))) T* Ptr;
    return *(Ptr)((Bytes)base + i * static_cast<uint32_t>(sizeof(T)));
}
__device__ __forceinline__ double2 load_at(const double2* base, uint32_t i) {
    typedef double V2 __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(1))) char* Bytes;
    const V2 v = *(const __attribute__((address_space(1))) V2*)((Bytes)base + i * 16u);
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ void store_at(double* base, uint32_t i, double v) {
    *(__attribute__((address_space(1))) double*)((__attribute__((address_space(1))) char*)base + i * 8u) = v;
}
__device__ __forceinline__ void store_at(double2* base, uint32_t i, double2 v) {
    typedef double V2 __attribute__((ext_vector_type(2)));
    V2 t;
    t.x = v.x;
    t.y = v.y;
    *(__attribute__((address_space(1))) V2*)((__attribute__((address_space(1))) char*)base + i * 16u) = t;
}

struct NoSync {
    __device__ __forceinline__ void operator()() const {}
};

// The LDS passes first..last-1 of `lines` lines at buf, in place.
template <int kMaxR, bool kInv>
__device__ __forceinline__ void lds_passes(const LinePlan& f, int first, int last, int lines, int stride, double2* buf,
                                           const double2* tw) {
    for (int s = first; s < last; s++) {
        const Where w = line::where_j_fast(f.per[s], lines);
        double2* b = buf + w.line * stride;
        auto ld = [&](int e) { return b[slot(e)]; };
        auto sync = [] { __syncthreads(); };
        auto st = [&](int e, double2 v) { b[slot(e)] = v; };
        if (s == 0) pass<kMaxR, kInv, true>(f, s, w, tw, ld, line::Same{}, sync, st);
        else pass<kMaxR, kInv, false>(f, s, w, tw, ld, line::Same{}, sync, st);
        __syncthreads();
    }
}

// zfwd: magnetisation (or raw reals) of pairs of z columns, one in the real
// and one in the imaginary parts -> z transform -> half spectrum in
// [x][kz][y] (magnetostatic_solver.cpp:121-151).  kSrc: what a column holds.
enum class Src { kRaw, kFm, kAll };

// What zfwd reads of a cell before its code is known.
template <Src kSrc>
struct CellIn {
    double m;
    uint32_t code;
    double m1, m2;
};
template <>
struct CellIn<Src::kRaw> {
    double m;
};
template <>
struct CellIn<Src::kFm> {
    double m;
    uint32_t code;
};

// The first pass of the z transforms takes radices up to this (z lines are
// planned so): its butterfly holds two columns' inputs per element.
constexpr int kMaxFirstZ = 8;

template <int kMaxR, Src kSrc>
__global__ void __launch_bounds__(kMaxThreads) zfwd_any_kernel(AnyPassArgs a) {
    extern __shared__ double2 smem[];
    const int c = blockIdx.z, x = blockIdx.y, y0 = blockIdx.x * a.pencils;
    const int nz = a.f.n;
    const int pairs = a.pencils > 1 ? a.pencils >> 1 : 1;
    double2* tw = smem;
    double2* buf = tw + nz;
    const int64_t plane = static_cast<int64_t>(x) * a.ny * nz;
    const bool fm = kSrc != Src::kAll || a.fm[c];
    const double* mc = (kSrc == Src::kRaw ? a.raw[c] : fm ? a.fm[c] : a.a1[c]) + plane;
    const double* a1c = a.a1[c] + plane;
    const double* a2c = a.a2[c] + plane;
    const uint32_t* code = a.code + plane;
    const double Ms1 = kSrc == Src::kRaw ? 0. : a.mats[0].Ms;   // the only material's, when there is one
    // columns past the last read the last one's cells and count as zero
    auto read = [&](int y, int k) {
        const uint32_t cell = static_cast<uint32_t>(min(y, a.ny - 1) * nz + k);
        CellIn<kSrc> in;
        if constexpr (kSrc == Src::kRaw) {
            in.m = load_at(mc, cell);
        } else {
            in.code = load_at(code, cell);
            in.m = load_at(mc, cell);
            if constexpr (kSrc == Src::kAll) {
                in.m1 = load_at(a1c, cell);
                in.m2 = load_at(a2c, cell);
            }
        }
        return in;
    };
    auto value = [&](const CellIn<kSrc>& in, int y) {
        double v = 0.;
        if constexpr (kSrc == Src::kRaw) {
            v = in.m;
        } else {
            const uint32_t mat = in.code & kMatMask;
            const DevMaterial* M = a.mats + (mat && a.nmat > 1 ? mat - 1 : 0);
            if constexpr (kSrc == Src::kAll) {
                if (in.code & kIsFM) v = M->Ms * in.m;
                else if (in.code & kIsAFM) v = M->aMs[0] * in.m1 + M->aMs[1] * in.m2;
            } else {
                const double Ms = a.nmat > 1 ? M->Ms : Ms1;
                v = in.code & kIsFM ? Ms * in.m : 0.;
            }
        }
        return y < a.ny ? v : 0.;
    };
    struct Pair {
        CellIn<kSrc> p, q;
    };
    {
        const Where w = line::where_j_fast(a.f.per[0], pairs);
        const int ya = y0 + w.line, yb = a.pencils > 1 ? ya + pairs : a.ny;
        double2* b = buf + w.line * a.stride;
        pass<kMaxR < kMaxFirstZ ? kMaxR : kMaxFirstZ, false, true>(
            a.f, 0, w, tw, [&](int e) { return Pair{read(ya, e), read(yb, e)}; },
            [&](const Pair& in, int) { return make_double2(value(in.p, ya), value(in.q, yb)); }, NoSync{},
            [&](int e, double2 v) { b[slot(e)] = v; });
    }
    load_table(tw, a.tw, nz);
    __syncthreads();
    lds_passes<kMaxR, false>(a.f, 1, a.f.count, pairs, a.stride, buf, tw);
    double2* out = a.spec + c * a.nh + static_cast<int64_t>(x) * a.nzh * a.ny;
    const int logq = a.pencils > 1 ? a.logp - 1 : 0;
    for (int idx = threadIdx.x; idx < pairs * a.nzh; idx += blockDim.x) {
        const int r = idx & (pairs - 1), kz = idx >> logq;
        const double2 Z = buf[r * a.stride + slot(kz)];
        const double2 Zm = buf[r * a.stride + slot(kz ? nz - kz : 0)];
        const uint32_t at = static_cast<uint32_t>(kz * a.ny + y0 + r);
        if (y0 + r < a.ny) store_at(out, at, make_double2((Z.x + Zm.x) * 0.5, (Z.y - Zm.y) * 0.5));
        if (a.pencils > 1 && y0 + r + pairs < a.ny)
            store_at(out, at + static_cast<uint32_t>(pairs), make_double2((Z.y + Zm.y) * 0.5, (Zm.x - Z.x) * 0.5));
    }
}

// y forward: [x][kz][y] (spec) -> [kz][y][x] (spec2, planes from kz0,
// component stride nhb); y inverse the other way.
template <int kMaxR, bool kInv>
__global__ void __launch_bounds__(kMaxThreads) y_any_kernel(AnyPassArgs a) {
    extern __shared__ double2 smem[];
    const int c = blockIdx.z, kz = a.kz0 + static_cast<int>(blockIdx.y), x0 = blockIdx.x * a.pencils;
    const int kb = kz - a.kzb0;
    const int ny = a.f.n, last = a.f.count - 1;
    double2* tw = smem;
    double2* buf = tw + ny;
    double2* spec = a.spec + c * a.nh + (static_cast<int64_t>(x0) * a.nzh + kz) * ny;
    double2* spec2 = a.spec2 + c * a.nhb + static_cast<int64_t>(kb) * ny * a.nx + x0;
    const uint32_t row = static_cast<uint32_t>(a.nzh) * static_cast<uint32_t>(ny), nx = static_cast<uint32_t>(a.nx);
    auto lines_of = [&](int s, bool line_fast) {
        return line_fast ? line::where_line_fast(static_cast<int>(a.f.per[s].d), a.logp)
                         : line::where_j_fast(a.f.per[s], a.pencils);
    };
    {
        Where w = lines_of(0, kInv);
        const uint32_t l = static_cast<uint32_t>(w.line);
        w.on = w.on && x0 + w.line < a.nx;
        double2* b = buf + w.line * a.stride;
        pass<kMaxR, kInv, true>(
            a.f, 0, w, tw,
            [&](int y) {
                const uint32_t e = static_cast<uint32_t>(y);
                return kInv ? load_at(spec2, e * nx + l) : load_at(spec, l * row + e);
            },
            line::Same{}, NoSync{}, [&](int e, double2 v) { b[slot(e)] = v; });
    }
    load_table(tw, a.tw, ny);
    __syncthreads();
    lds_passes<kMaxR, kInv>(a.f, 1, last, a.pencils, a.stride, buf, tw);
    {
        Where w = lines_of(last, !kInv);
        const uint32_t l = static_cast<uint32_t>(w.line);
        w.on = w.on && x0 + w.line < a.nx;
        const double2* b = buf + w.line * a.stride;
        pass<kMaxR, kInv, false>(
            a.f, last, w, tw, [&](int e) { return b[slot(e)]; }, line::Same{}, NoSync{},
            [&](int y, double2 v) {
                const uint32_t e = static_cast<uint32_t>(y);
                if (kInv) store_at(spec, l * row + e, v);
                else store_at(spec2, e * nx + l, v);
            });
    }
}

// x forward, the tensor product (magnetostatic_solver.cpp:163-177) and x
// inverse in place on [kz][y][x] (spec2); conv = 0: forward transform of
// component 0 only (tensor set-up).
template <int kMaxR>
__global__ void __launch_bounds__(kMaxThreads) xconv_any_kernel(AnyPassArgs a) {
    extern __shared__ double2 smem[];
    const int kz = a.kz0 + static_cast<int>(blockIdx.y), y0 = blockIdx.x * a.pencils;
    const int kb = kz - a.kzb0;
    const int nx = a.f.n, last = a.f.count - 1;
    const int lines = (a.conv ? 3 : 1) * a.pencils;
    double2* tw = smem;
    double2* buf = tw + nx;
    auto row = [&](int line) {
        return a.spec2 + (line >> a.logp) * a.nhb +
               (static_cast<int64_t>(kb) * a.ny + y0 + (line & (a.pencils - 1))) * nx;
    };
    auto inside = [&](int line) { return y0 + (line & (a.pencils - 1)) < a.ny; };
    // Tensor spectra of one k-point in the order xx, yy, zz, xy, yz, zx, yx,
    // zy, xz; the adjoint convolution uses N^T with conjugated spectra.  A
    // thread's first point is read with the magnetisation spectra, before the
    // transforms.
    double kr[9];
    float ki[9];
    auto load_tensor = [&](int idx) {
        const int r = line::div(a.nn, idx), x = idx - r * nx;
        if (idx >= a.pencils * nx || y0 + r >= a.ny) return;
        const int64_t g = (static_cast<int64_t>(kz) * a.ny + y0 + r) * nx + x;
#pragma unroll
        for (int q = 0; q < 9; q++) {
            const int t = a.adjoint ? (q < 3 ? q : (q < 6 ? q + 3 : q - 3)) : q;
            // the tensor is streamed once per convolution
            kr[q] = __builtin_nontemporal_load(&a.kre[t * a.nh + g]);
            ki[q] = __builtin_nontemporal_load(&a.kim[t * a.nh + g]);
        }
    };
    if (a.conv) load_tensor(threadIdx.x);
    {
        Where w = line::where_j_fast(a.f.per[0], lines);
        w.on = w.on && inside(w.line);
        const double2* in = row(w.line);
        double2* b = buf + w.line * a.stride;
        pass<kMaxR, false, true>(
            a.f, 0, w, tw, [&](int e) { return in[e]; }, line::Same{}, NoSync{}, [&](int e, double2 v) { b[slot(e)] = v; });
    }
    load_table(tw, a.tw, nx);
    __syncthreads();
    lds_passes<kMaxR, false>(a.f, 1, a.f.count, lines, a.stride, buf, tw);
    if (!a.conv) {
        for (int idx = threadIdx.x; idx < lines * nx; idx += blockDim.x) {
            const int l = line::div(a.nn, idx), x = idx - l * nx;
            if (inside(l)) row(l)[x] = buf[l * a.stride + slot(x)];
        }
        return;
    }
    for (int idx = threadIdx.x; idx < a.pencils * nx; idx += blockDim.x) {
        const int r = line::div(a.nn, idx), x = idx - r * nx;
        if (y0 + r >= a.ny) continue;
        if (idx != static_cast<int>(threadIdx.x)) load_tensor(idx);
        double2 K[9];
#pragma unroll
        for (int q = 0; q < 9; q++) {
            const double im = static_cast<double>(ki[q]);
            K[q] = make_double2(kr[q], a.adjoint ? -im : im);
        }
        double2* bx = buf + r * a.stride + slot(x);
        double2* by = bx + a.pencils * a.stride;
        double2* bz = by + a.pencils * a.stride;
        const double2 mx = *bx, my = *by, mz = *bz;
        auto sum = [&](double2 p, double2 q, double2 s) {
            return make_double2((p.x + q.x + s.x) * a.rden, (p.y + q.y + s.y) * a.rden);
        };
        *bx = sum(line::mul(mx, K[0]), line::mul(my, K[3]), line::mul(mz, K[8]));
        *by = sum(line::mul(my, K[1]), line::mul(mz, K[4]), line::mul(mx, K[6]));
        *bz = sum(line::mul(mz, K[2]), line::mul(mx, K[5]), line::mul(my, K[7]));
    }
    __syncthreads();
    lds_passes<kMaxR, true>(a.f, 0, last, lines, a.stride, buf, tw);
    {
        Where w = line::where_j_fast(a.f.per[last], lines);
        w.on = w.on && inside(w.line);
        double2* out = row(w.line);
        const double2* b = buf + w.line * a.stride;
        pass<kMaxR, true, false>(
            a.f, last, w, tw, [&](int e) { return b[slot(e)]; }, line::Same{}, NoSync{}, [&](int e, double2 v) { out[e] = v; });
    }
}

// z complex-to-real inverse: Hermitian extension of the half spectra
// [x][kz][y] of two columns as one complex line, inverse transform, real
// parts the one column and imaginary parts the other (cuFFT Z2D semantics:
// the imaginary parts of the self-conjugate bins are ignored).
template <int kMaxR>
__global__ void __launch_bounds__(kMaxThreads) zinv_any_kernel(AnyPassArgs a) {
    extern __shared__ double2 smem[];
    const int c = blockIdx.z, x = blockIdx.y, y0 = blockIdx.x * a.pencils;
    const int nz = a.f.n, last = a.f.count - 1;
    const int pairs = a.pencils > 1 ? a.pencils >> 1 : 1;
    const int logq = a.pencils > 1 ? a.logp - 1 : 0;
    double2* tw = smem;
    double2* buf = tw + nz;
    struct Pair {
        double2 A, B;
    };
    {
        const Where w = line::where_line_fast(static_cast<int>(a.f.per[0].d), logq);
        const double2* in = a.spec + c * a.nh + static_cast<int64_t>(x) * a.nzh * a.ny;
        // columns past the last read the last one's and count as zero
        const int ya = y0 + w.line, yb = a.pencils > 1 ? ya + pairs : a.ny;
        const bool ona = ya < a.ny, onb = yb < a.ny;
        const uint32_t ra = static_cast<uint32_t>(min(ya, a.ny - 1)), rb = static_cast<uint32_t>(min(yb, a.ny - 1));
        double2* b = buf + w.line * a.stride;
        pass<kMaxR < kMaxFirstZ ? kMaxR : kMaxFirstZ, true, true>(
            a.f, 0, w, tw,
            [&](int k) {
                const uint32_t at = static_cast<uint32_t>((2 * k > nz ? nz - k : k) * a.ny);
                return Pair{load_at(in, at + ra), load_at(in, at + rb)};
            },
            [&](const Pair& p, int k) {
                double2 A = ona ? p.A : make_double2(0., 0.), B = onb ? p.B : make_double2(0., 0.);
                if (k == 0 || 2 * k == nz) { A.y = 0.; B.y = 0.; }
                return 2 * k > nz ? make_double2(A.x + B.y, B.x - A.y) : make_double2(A.x - B.y, A.y + B.x);
            },
            NoSync{}, [&](int e, double2 v) { b[slot(e)] = v; });
    }
    load_table(tw, a.tw, nz);
    __syncthreads();
    lds_passes<kMaxR, true>(a.f, 1, last, pairs, a.stride, buf, tw);
    {
        Where w = line::where_j_fast(a.f.per[last], pairs);
        const double2* b = buf + w.line * a.stride;
        double* o = a.out[c] + (static_cast<int64_t>(x) * a.ny + y0) * nz;
        // a pair without a second column writes its first one twice, which
        // keeps the stores free of branches
        w.on = w.on && y0 + w.line < a.ny;
        const bool two = a.pencils > 1 && y0 + w.line + pairs < a.ny;
        const uint32_t first = static_cast<uint32_t>(w.line * nz);
        const uint32_t second = two ? first + static_cast<uint32_t>(pairs * nz) : first;
        pass<kMaxR, true, false>(
            a.f, last, w, tw, [&](int e) { return b[slot(e)]; }, line::Same{}, NoSync{},
            [&](int k, double2 v) {
                store_at(o, first + static_cast<uint32_t>(k), v.x);
                store_at(o, second + static_cast<uint32_t>(k), two ? v.y : v.x);
            });
    }
}

int ilog2(int n) {
    int l = 0;
    while ((1 << l) < n) l++;
    return l;
}

}  // namespace

// Dynamic LDS beyond 64 KB (up to the 160 KB of a gfx950 CU) is allowed
// per kernel; a refusal of the attribute is left to the launch to report.
static void allow_lds(const void* fn, size_t lds) {
    if (lds <= 64 * 1024) return;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)) != hipSuccess)
        (void)hipGetLastError();
}

// Lines per workgroup: a workgroup's threads take one butterfly each, at
// most kThreads of them as long as that leaves two lines, and the launch
// keeps kFill workgroups (two per CU) when it can while runs stay at kRun
// lines (64 B of the transposed side).  `cap` bounds the lines at the
// extent they run along.
static int pick_lines(const LinePlan& f, int per_line, int cap, int64_t others) {
    constexpr int kThreads = 256, kRun = 4, kMost = 16;
    constexpr int64_t kFill = 512;
    int p = 1;
    while (p * 2 <= kMost && p < cap && p * 2 * per_line * f.width <= kThreads) p *= 2;
    while (p > kRun && (cap + p - 1) / p * others < kFill) p /= 2;
    return p;
}

template <class Kernel>
static hipError_t launch(Kernel k, const AnyPassArgs& a, dim3 grid, int threads, size_t lds, hipStream_t s) {
    allow_lds(reinterpret_cast<const void*>(k), lds);
    hipLaunchKernelGGL(k, grid, dim3(static_cast<unsigned>(threads)), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_any_pass(AnyPass kind, AnyPassArgs a, int comps, int planes, hipStream_t s) {
    const LinePlan& f = a.f;
    const bool z = kind == AnyPass::kZFwd || kind == AnyPass::kZInv, xc = kind == AnyPass::kXConv;
    int lines;
    if (z) {
        lines = pick_lines(f, 1, (a.ny + 1) / 2, static_cast<int64_t>(a.nx) * comps);
        a.pencils = a.ny > 1 ? 2 * lines : 1;
    } else {
        const int mult = xc && a.conv ? 3 : 1;
        a.pencils = pick_lines(f, mult, xc ? a.ny : a.nx, static_cast<int64_t>(planes) * (xc ? 1 : comps));
        lines = mult * a.pencils;
    }
    a.logp = ilog2(a.pencils);
    a.stride = (f.n + f.n / 16) | 1;
    a.nn = FastDiv{static_cast<uint32_t>(f.n), static_cast<uint32_t>(((uint64_t{1} << 32) + f.n - 1) / f.n)};
    // The product takes up to 256 threads, whether or not the butterflies do,
    // so that most of a workgroup's tensor reads are in flight at once (96x128x32:
    // 17 us a launch, 22 with up to 512 threads or with the butterflies' 192).
    const int width = xc && a.conv ? std::max(lines * f.width, std::min(a.pencils * f.n, 256)) : lines * f.width;
    const int threads = (width + 63) / 64 * 64;
    const size_t lds = sizeof(double2) * (static_cast<size_t>(f.n) + static_cast<size_t>(lines) * a.stride);
    if (threads > kMaxThreads || lds > 160 * 1024 || f.count < 2 || (z && f.r[0] > kMaxFirstZ)) return hipErrorInvalidValue;
    const int across = z || xc ? a.ny : a.nx;
    const dim3 grid(static_cast<unsigned>((across + a.pencils - 1) / a.pencils),
                    static_cast<unsigned>(z ? a.nx : planes), static_cast<unsigned>(xc ? 1 : comps));
    const bool small = f.maxr <= 8;
    switch (kind) {
    case AnyPass::kZFwd:
        if (a.raw_in)
            return small ? launch(zfwd_any_kernel<8, Src::kRaw>, a, grid, threads, lds, s)
                         : launch(zfwd_any_kernel<16, Src::kRaw>, a, grid, threads, lds, s);
        if (!a.a1[0])
            return small ? launch(zfwd_any_kernel<8, Src::kFm>, a, grid, threads, lds, s)
                         : launch(zfwd_any_kernel<16, Src::kFm>, a, grid, threads, lds, s);
        return small ? launch(zfwd_any_kernel<8, Src::kAll>, a, grid, threads, lds, s)
                     : launch(zfwd_any_kernel<16, Src::kAll>, a, grid, threads, lds, s);
    case AnyPass::kYFwd:
        return small ? launch(y_any_kernel<8, false>, a, grid, threads, lds, s)
                     : launch(y_any_kernel<16, false>, a, grid, threads, lds, s);
    case AnyPass::kYInv:
        return small ? launch(y_any_kernel<8, true>, a, grid, threads, lds, s)
                     : launch(y_any_kernel<16, true>, a, grid, threads, lds, s);
    case AnyPass::kXConv:
        return small ? launch(xconv_any_kernel<8>, a, grid, threads, lds, s) : launch(xconv_any_kernel<16>, a, grid, threads, lds, s);
    case AnyPass::kZInv:
        return small ? launch(zinv_any_kernel<8>, a, grid, threads, lds, s) : launch(zinv_any_kernel<16>, a, grid, threads, lds, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace gf
