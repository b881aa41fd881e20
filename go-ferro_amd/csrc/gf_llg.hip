// gf_llg.hip — fused LLG RK4 stage kernels for gfx950 (FP64).
//
// One launch per RK stage does what the reference spreads over get_dm_RKs,
// get_dm (at stage 4) and update_m_RKs / update_m
// (magnetic_solver.cpp:3-229, 1449-1457, 1515-1636;
//  magnetic_AFM_solver.cpp:3-430, 1715-1834):
//   stage 1:  k = f(m);      next = m + k/2;  acc = k/6
//   stage 2:  k = f(s2);     next = m + k/2;  acc = acc + k/3
//   stage 3:  k = f(s3);     next = m + k;    acc = acc + k/3
//   stage 4:  k = f(s4);     m = m + (acc + k/6)
// The accumulator is summed in the reference's order
// (((k1/6 + k2/3) + k3/3) + k4/6), the weights applied as products with the
// rounded reciprocals (within about an ulp of the reference's quotients);
// the four k-arrays and the separate combine/update/copy launches disappear.  The
// stencil store is read-only within a stage and the next store goes to the
// other buffer, so physics that share a stage still see the old store.
#include "gf_fm_dev.h"

namespace gf {

namespace {

// Material records the lean fused stage copies into LDS (about 0.9 KB each),
// and the set-up loads per thread of a 256-thread workgroup: up to
// kMatWordsPerThread words of those records, and the field spectrum in
// chunks of kSetupChunk complex values.
constexpr int kLeanMats = 8;
constexpr int kMatWordsPerThread = 4;
constexpr int kSetupChunk = 4;
static_assert(kLeanMats * sizeof(DevMaterial) / sizeof(double) <= kMatWordsPerThread * 256,
              "the lean stage's material records must fit the set-up loads of 256 threads");

template <class I, bool kMixed>
__global__ void __launch_bounds__(256) mag_stage_kernel(StageArgs) {
    const StageArgs& a = launch_arg<StageArgs>();
    const I n = static_cast<I>(a.nx * a.ny * a.nz);
    const I id = static_cast<I>(blockIdx.x) * static_cast<I>(blockDim.x) + static_cast<I>(threadIdx.x);
    if (id >= n) return;
    fm_point<I, true, kMixed>(a, id);
}

// The same over a list of the FM cells: a layered magnet fills whole
// waves instead of loading the inputs of every non-magnetic cell first.  The
// list is of 32-bit indices on every grid that has one (up to 2^32 cells).
template <class I, bool kMixed>
__global__ void __launch_bounds__(256) mag_stage_list_kernel(StageArgs, const uint32_t* ids, I count) {
    const StageArgs& a = launch_arg<StageArgs>();
    const I t = static_cast<I>(blockIdx.x) * static_cast<I>(blockDim.x) + static_cast<I>(threadIdx.x);
    if (t >= count) return;
    fm_point<I, false, kMixed>(a, static_cast<I>(ldu(ids, t)));
}

// The FM stage fused with the z transforms of the FFT magnetostatics, for
// contexts whose magnetisation is FM only.  A workgroup owns P whole z
// columns (fixed x, consecutive y): it rebuilds their static field from
// the H z-spectrum (inverse real transform in LDS, two real columns per
// complex transform, the imaginary parts of the self-conjugate bins
// ignored as a complex-to-real transform does), runs the stage on every
// cell, and forward-transforms Ms m of the new store into the M z-spectrum.
// The three components are transformed together.  Column p < P/2 lives in
// the real parts and column p + P/2 in the imaginary parts of transform p;
// the inverse leaves sample k at bit-reversed position, which is where the
// forward transform wants its input, so each cell's H is read and its M
// written in the same LDS slot.  Both spectra use the layout [x][kz][y] of
// the separate z passes (gf_fft.hip), so the y and x passes are unchanged.
// Workgroups are ordered so that each XCD takes a contiguous range of x
// planes, keeping stencil neighbours in its L2.  The lean form also copies
// the material records into LDS (at most kLeanMats of them).
template <bool kHspec, bool kLean, bool kMixed, class I>
__global__ void __launch_bounds__(256) mag_stage_fused_kernel(StageArgs a, FusedZArgs f) {
    extern __shared__ double2 fsm[];
    const int nz = static_cast<int>(a.nz), ny = static_cast<int>(a.ny);
    const int P = f.P, lognz = f.lognz, nzh = f.nzh;
    const int pairs = P > 1 ? P >> 1 : 1;
    double2* tw = fsm;
    double2* cbuf = tw + (nz >> 1);          // [3][pairs][nz], element i at slot fpad(i)
    DevMaterial* ltab = reinterpret_cast<DevMaterial*>(cbuf + fft_lds_elems(3 * pairs * nz));
    const int tid = threadIdx.x, bd = blockDim.x;
    const unsigned L = xcd_group(blockIdx.x, gridDim.x);
    const int gpx = ny / P;
    const int x = static_cast<int>(L) / gpx, y0 = (static_cast<int>(L) % gpx) * P;
    const int cells = P * nz;
    // The set-up loads (twiddles, material records, the field spectrum in
    // chunks of kSetupChunk elements per thread) are issued before any of
    // them is written to LDS, so that together they cost one memory round
    // trip per chunk rather than one each.
    const int ntw = nz >> 1;
    const int words = kLean ? a.nmat * static_cast<int>(sizeof(DevMaterial) / sizeof(double)) : 0;
    const double2 twv = tid < ntw ? f.tw[tid] : make_double2(0., 0.);
    double mw[kMatWordsPerThread];
#pragma unroll
    for (int u = 0; u < kMatWordsPerThread; u++) {
        const int t = tid + u * bd;
        mw[u] = t < words ? ldd(reinterpret_cast<const double*>(a.mats), static_cast<uint32_t>(t)) : 0.;
    }
    bool setup_stored = false;
    auto store_setup = [&]() {
        if (tid < ntw) tw[tid] = twv;
        for (int j = tid + bd; j < ntw; j += bd) tw[j] = f.tw[j];
#pragma unroll
        for (int u = 0; u < kMatWordsPerThread; u++) {
            const int t = tid + u * bd;
            if (t < words) reinterpret_cast<double*>(ltab)[t] = mw[u];
        }
        setup_stored = true;
    };
    if (kHspec) {
        const int per = pairs * nzh, tot = 3 * per;
        for (int t0 = 0; t0 < tot; t0 += kSetupChunk * bd) {
            double2 A[kSetupChunk], B[kSetupChunk];
#pragma unroll
            for (int u = 0; u < kSetupChunk; u++) {
                const int t = t0 + u * bd + tid;
                A[u] = make_double2(0., 0.);
                B[u] = make_double2(0., 0.);
                if (t < tot) {
                    const int c = t / per, w = t - c * per;
                    const int p = w % pairs, kz = w / pairs;
                    const int64_t row = (static_cast<int64_t>(x) * nzh + kz) * ny + y0;
                    const double2* in = f.hspec + c * f.nh;
                    A[u] = in[row + p];
                    if (P > 1) B[u] = in[row + p + pairs];
                }
            }
            if (!setup_stored) store_setup();
#pragma unroll
            for (int u = 0; u < kSetupChunk; u++) {
                const int t = t0 + u * bd + tid;
                if (t < tot) {
                    const int c = t / per, w = t - c * per;
                    const int p = w % pairs, kz = w / pairs;
                    double2 Av = A[u], Bv = B[u];
                    if (kz == 0 || 2 * kz == nz) { Av.y = 0.; Bv.y = 0.; }
                    const int cb = (c * pairs + p) * nz;
                    cbuf[fpad(cb + kz)] = make_double2(Av.x - Bv.y, Av.y + Bv.x);
                    if (kz > 0 && 2 * kz < nz) cbuf[fpad(cb + nz - kz)] = make_double2(Av.x + Bv.y, Bv.x - Av.y);
                }
            }
        }
        __syncthreads();
        ifft_dif(cbuf, 3 * pairs, lognz, tw);
    } else {
        store_setup();
        for (int t = threadIdx.x; t < 3 * cells; t += blockDim.x) {
            const int c = t / cells, w = t - c * cells;
            const int col = w >> lognz, k = w & (nz - 1);
            const double h = a.hstat[c][(static_cast<int64_t>(x) * ny + y0 + col) * nz + k];
            const int p = col < pairs ? col : col - pairs;
            double* slot2 = reinterpret_cast<double*>(cbuf + fpad((c * pairs + p) * nz + fft_bitrev(k, lognz)));
            slot2[col < pairs ? 0 : 1] = h;
        }
        __syncthreads();
    }
    for (int w = threadIdx.x; w < cells; w += blockDim.x) {
        const int col = w >> lognz, k = w & (nz - 1);
        const int y = y0 + col;
        const int p = col < pairs ? col : col - pairs;
        const int part = col < pairs ? 0 : 1;
        const int pos = p * nz + fft_bitrev(k, lognz);
        double* h0 = reinterpret_cast<double*>(cbuf + fpad(pos)) + part;
        double* h1 = reinterpret_cast<double*>(cbuf + fpad(pairs * nz + pos)) + part;
        double* h2 = reinterpret_cast<double*>(cbuf + fpad(2 * pairs * nz + pos)) + part;
        const I id = (static_cast<I>(x) * static_cast<I>(ny) + static_cast<I>(y)) * static_cast<I>(nz) + static_cast<I>(k);
        FmIn in;
        fm_load<I, true, kMixed>(a, id, static_cast<I>(x), static_cast<I>(y), static_cast<I>(k), in);
        double mx = 0., my = 0., mz = 0.;
        if (in.own & kIsFM) {
            double n0, n1, n2;
            double Ms;
            if (kLean) {
                LMat* tab = (LMat*)ltab;
                fm_cell<kLean, kMixed, I>(a, tab, in, id, static_cast<I>(k), *h0, *h1, *h2, n0, n1, n2);
                Ms = tab[(in.own & kMatMask) - 1].Ms;
            } else {
                fm_cell<kLean, kMixed, I>(a, (GMat*)a.mats, in, id, static_cast<I>(k), *h0, *h1, *h2, n0, n1, n2);
                Ms = mat_of(a.mats, in.own).Ms;
            }
            mx = Ms * n0; my = Ms * n1; mz = Ms * n2;
        }
        *h0 = mx; *h1 = my; *h2 = mz;
        if (P == 1) {
            // a lone column: the imaginary parts of the forward input are zero
            h0[1] = 0.; h1[1] = 0.; h2[1] = 0.;
        }
    }
    __syncthreads();
    fft_dit(cbuf, 3 * pairs, lognz, tw);
    const int per = pairs * nzh;
    for (int t = threadIdx.x; t < 3 * per; t += blockDim.x) {
        const int c = t / per, u = t - c * per;
        const int p = u % pairs, kz = u / pairs;
        const int cb = (c * pairs + p) * nz;
        const double2 Z = cbuf[fpad(cb + kz)];
        const double2 Zm = cbuf[fpad(cb + ((nz - kz) & (nz - 1)))];
        const int64_t row = (static_cast<int64_t>(x) * nzh + kz) * ny + y0;
        double2* out = f.mspec + c * f.nh;
        if (P > 1) {
            out[row + p] = make_double2((Z.x + Zm.x) * 0.5, (Z.y - Zm.y) * 0.5);
            out[row + p + pairs] = make_double2((Z.y + Zm.y) * 0.5, (Zm.x - Z.x) * 0.5);
        } else {
            out[row + p] = Z;
        }
    }
}

// One sublattice of one AFM cell: the two sublattices of a stage read only
// stage-(s-1) stores, so they run as independent threads.  Every global
// input of the sublattice is loaded before the cell's code is known (all
// indices are in bounds), as for the FM cell, so one memory round trip
// feeds the cell.
template <class I, bool kLanes, bool kMixed>
__device__ __forceinline__ void afm_point(const AfmStageArgs& a, I id, int sub) {
    const I ny = static_cast<I>(a.ny), nz = static_cast<I>(a.nz);
    I x, y, z;
    cell_xyz(a.div, id, ny, nz, x, y, z);
    const P3 s1 = {{a.store1[0], a.store1[1], a.store1[2]}}, s2 = {{a.store2[0], a.store2[1], a.store2[2]}};
    const P3 st = sub == 0 ? s1 : s2;
    const P3 other = sub == 0 ? s2 : s1;
    const double* const* base = sub == 0 ? a.base1 : a.base2;
    double* const* acc = sub == 0 ? a.acc1 : a.acc2;
    double* const* out = sub == 0 ? a.out1 : a.out2;
    const uint32_t own = ldu(a.code, id);
    const double c3[3] = {ldd(st.p[0], id), ldd(st.p[1], id), ldd(st.p[2], id)};
    const double mgx = c3[0], mgy = c3[1], mgz = c3[2];
    const I nx = static_cast<I>(a.nx);
    double v[6][3];
    uint32_t cd[6];
    if (kLanes) gather6_lanes_load<kMixed, I>(st, a.code, x, y, z, nx, ny, nz, v, cd);
    else gather6<kMixed, I>(st, a.code, x, y, z, nx, ny, nz, v, cd);
    const double o0 = ldd(other.p[0], id), o1 = ldd(other.p[1], id), o2 = ldd(other.p[2], id);
    // a null Hstat is zero (no statics, nothing uploaded)
    const bool hs = a.hstat[0] != nullptr;
    const double hs0 = hs ? ldd(a.hstat[0], id) : 0., hs1 = hs ? ldd(a.hstat[1], id) : 0.;
    const double hs2 = hs ? ldd(a.hstat[2], id) : 0.;
    // at stage 1 the stage store is m itself: read it once
    const bool same = base[0] == st.p[0] && base[1] == st.p[1] && base[2] == st.p[2];
    double mb[3], ac[3];
    mb[0] = same ? mgx : ldd_nt(base[0], id);
    mb[1] = same ? mgy : ldd_nt(base[1], id);
    mb[2] = same ? mgz : ldd_nt(base[2], id);
    for (int c = 0; c < 3; c++) ac[c] = a.stage > 1 ? ldd_nt(acc[c], id) : 0.;
    if (kLanes) gather6_lanes_shift<kMixed, I>(z, nz, c3, own, v, cd);
    if (!(own & kIsAFM)) return;
    GMat& M = mat_of(a.mats, own);
    double mx = mgx, my = mgy, mz = mgz;
    if (a.rotate) rot(a.Tg2c, mgx, mgy, mgz, mx, my, mz);
    const Stencil s = magnet_stencil<false, kMixed>(c3, v, cd, (GMat*)a.mats, own, kAfmSurfShift, sub, a.idx, a.idy,
                                                    a.idz, M.aAex[sub], M.aAex_self[sub], 0.);
    // uniaxial anisotropy 2K1 (u.m) u (magnetic_AFM_solver.cpp:148-154)
    const double udotm = mx * M.u[0] + my * M.u[1] + mz * M.u[2];
    const double hac0 = 2. * M.aK1n[sub] * udotm * M.u[0];
    const double hac1 = 2. * M.aK1n[sub] * udotm * M.u[1];
    const double hac2 = 2. * M.aK1n[sub] * udotm * M.u[2];
    double ha0 = hac0, ha1 = hac1, ha2 = hac2;
    if (a.rotate) rot(a.Tc2g, hac0, hac1, hac2, ha0, ha1, ha2);
    // magnetoelastic (magnetic_AFM_solver.cpp:89-96, 156-162), exchange,
    // inter-sublattice coupling and drive (:170-200)
    double H0 = hs0 + ha0;
    double H1 = hs1 + ha1;
    double H2 = hs2 + ha2;
    if (a.strain[0]) {
        double he0, he1, he2;
        magnetoelastic(a.strain, a.strain0, id, -1., M.aB1n[sub], M.aB2n[sub], mx, my, mz, a.rotate, a.Tc2g, he0, he1, he2);
        H0 = H0 + he0;
        H1 = H1 + he1;
        H2 = H2 + he2;
    }
    H0 = H0 + M.aExch[sub] * s.ex[0] + M.aJ[sub] * o0 + a.hext[0];
    H1 = H1 + M.aExch[sub] * s.ex[1] + M.aJ[sub] * o1 + a.hext[1];
    H2 = H2 + M.aExch[sub] * s.ex[2] + M.aJ[sub] * o2 + a.hext[2];
    if (a.hcell[0]) {
        // electrodynamic back-action (magnetic_AFM_solver.cpp:222-226)
        H0 = H0 + ldd(a.hcell[0], id);
        H1 = H1 + ldd(a.hcell[1], id);
        H2 = H2 + ldd(a.hcell[2], id);
    }
    const double px = mgy * H2 - mgz * H1, py = mgz * H0 - mgx * H2, pz = mgx * H1 - mgy * H0;
    const double qx = mgy * pz - mgz * py, qy = mgz * px - mgx * pz, qz = mgx * py - mgy * px;
    const double k0 = M.aPrecess[sub] * px + M.aAlphaPrecess[sub] * qx;
    const double k1 = M.aPrecess[sub] * py + M.aAlphaPrecess[sub] * qy;
    const double k2 = M.aPrecess[sub] * pz + M.aAlphaPrecess[sub] * qz;
    double* const* dmo = sub == 0 ? a.dm_out1 : a.dm_out2;
    if (dmo[0]) {
        std_(dmo[0], id, k0); std_(dmo[1], id, k1); std_(dmo[2], id, k2);
    }
    rk_store(a.stage, id, 0, k0, mb[0], ac[0], acc, out);
    rk_store(a.stage, id, 1, k1, mb[1], ac[1], acc, out);
    rk_store(a.stage, id, 2, k2, mb[2], ac[2], acc, out);
}

// Workgroup b serves cell block (b / 16) * 8 + b % 8 and sublattice
// (b / 8) % 2: the two sublattices of a cell block land on the same XCD
// (workgroups are dealt to the 8 XCDs round-robin) one dispatch round
// apart, so the second finds the shared reads (code, Hstat, the other
// sublattice's store) in that XCD's L2.  Over one material the by-value argument
// is the faster one (64x64x32: 36.3 us a step, 37.9 through launch_arg).
template <class I, bool kMixed>
__global__ void __launch_bounds__(256) afm_stage_kernel(AfmStageArgs byval) {
    const AfmStageArgs& a = kMixed ? launch_arg<AfmStageArgs>() : byval;
    const unsigned b = blockIdx.x;
    const unsigned blk = (b >> 4) * 8u + (b & 7u);
    const int sub = static_cast<int>((b >> 3) & 1u);
    const I n = static_cast<I>(a.nx * a.ny * a.nz);
    const I id = static_cast<I>(blk) * static_cast<I>(blockDim.x) + static_cast<I>(threadIdx.x);
    if (id >= n) return;
    afm_point<I, true, kMixed>(a, id, sub);
}

// Batched stages: one launch covers every instance of a batch.  The stage
// arguments of instance i and stage s live in device memory at
// items[4*i + s - 1]; workgroup slot b (of L.total slots) serves instance
// L.item[b], the chunk of L.cpt * blockDim.x cells starting at
// (b - L.block0[instance]) * L.cpt * blockDim.x, one cell per thread per
// pass.  A grid smaller than L.total walks the slots with a stride of
// gridDim.x.
template <class I, bool kMixed>
__global__ void __launch_bounds__(256) mag_batch_kernel(const StageArgs* __restrict__ items, BatchLaunch L, int stage) {
    for (uint32_t b = blockIdx.x; b < L.total; b += gridDim.x) {
        const uint32_t inst = L.item[b];
        const StageArgs& a = items[4 * inst + stage - 1];
        const I n = static_cast<I>(a.nx * a.ny * a.nz);
        const I chunk = static_cast<I>(L.cpt) * static_cast<I>(blockDim.x);
        const I first = static_cast<I>(b - L.block0[inst]) * chunk + static_cast<I>(threadIdx.x);
        for (int j = 0; j < L.cpt; j++) {
            const I id = first + static_cast<I>(j) * static_cast<I>(blockDim.x);
            if (id < n) fm_point<I, true, kMixed>(a, id);
        }
    }
}

// Work item w of 2 * ceil(total / 8) * 8: slot (w / 16) * 8 + w % 8 and
// sublattice (w / 8) % 2, so that the two sublattices of a slot run on one
// XCD one dispatch round apart (see afm_stage_kernel).
// kOne: one work item per workgroup and one cell per thread (no loops).
template <class I, bool kOne, bool kMixed>
__global__ void __launch_bounds__(256) afm_batch_kernel(const AfmStageArgs* __restrict__ items, BatchLaunch L,
                                                         int stage) {
    const uint32_t work = 2u * ((L.total + 7u) / 8u * 8u);
    if (kOne) {
        const uint32_t w = blockIdx.x;
        const uint32_t b = (w >> 4) * 8u + (w & 7u);
        if (w >= work || b >= L.total) return;
        const uint32_t inst = L.item[b];
        const AfmStageArgs& a = items[4 * inst + stage - 1];
        const I n = static_cast<I>(a.nx * a.ny * a.nz);
        const I id = static_cast<I>(b - L.block0[inst]) * static_cast<I>(blockDim.x) + static_cast<I>(threadIdx.x);
        if (id < n) afm_point<I, true, kMixed>(a, id, static_cast<int>((w >> 3) & 1u));
        return;
    }
    for (uint32_t w = blockIdx.x; w < work; w += gridDim.x) {
        const uint32_t b = (w >> 4) * 8u + (w & 7u);
        const int sub = static_cast<int>((w >> 3) & 1u);
        if (b >= L.total) continue;
        const uint32_t inst = L.item[b];
        const AfmStageArgs& a = items[4 * inst + stage - 1];
        const I n = static_cast<I>(a.nx * a.ny * a.nz);
        const I chunk = static_cast<I>(L.cpt) * static_cast<I>(blockDim.x);
        const I first = static_cast<I>(b - L.block0[inst]) * chunk + static_cast<I>(threadIdx.x);
        for (int j = 0; j < L.cpt; j++) {
            const I id = first + static_cast<I>(j) * static_cast<I>(blockDim.x);
            // lane gathers cost this loop a wave of occupancy
            if (id < n) afm_point<I, false, kMixed>(a, id, sub);
        }
    }
}

// Per-instance clock of a batch: t += dt (global.cpp:513-549), then the
// sinusoidal drive at each stage time t - dt, t - dt/2, t - dt/2, t
// (magnetic_solver.cpp:1834-1861, magnetic_AFM_solver.cpp:61-64) written
// into the stage arguments of both magnet kinds.
// A batch without FM (or AFM) instances has no table of that kind: its
// pointer is null and is not written.
__global__ void __launch_bounds__(256) batch_clock_kernel(BatchClock* clk, StageArgs* fm, AfmStageArgs* afm,
                                                           int count) {
    const int i = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= count) return;
    const BatchClock c = clk[i];
    const double t = c.t + c.dt;
    clk[i].t = t;
    for (int s = 1; s <= 4; s++) {
        const double ts = s == 1 ? t - c.dt : (s == 4 ? t : t - c.dt * 0.5);
        for (int k = 0; k < 3; k++) {
            const double h = c.stat[k] + c.altr[k] * sin(2. * kPi * c.freq[k] * ts);
            if (fm) fm[4 * i + s - 1].hext[k] = h;
            if (afm) afm[4 * i + s - 1].hext[k] = h;
        }
    }
}

// update_prescribed_m (magnetic_solver.cpp:1937-1957): the FM cells of the
// bottom layer k = 0 take the cone value v.
__global__ void __launch_bounds__(256) prescribe_plane_kernel(double* m0, double* m1, double* m2,
                                                              const uint32_t* code, int64_t nxy, int64_t nz,
                                                              double v0, double v1, double v2) {
    const int64_t col = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (col >= nxy) return;
    const int64_t id = col * nz;
    if (!(code[id] & kIsFM)) return;
    m0[id] = v0; m1[id] = v1; m2[id] = v2;
}

// Per-block partial sums of three fields; block b writes partial[3*b + c].
__global__ void __launch_bounds__(256) sum3_kernel(const double* f0, const double* f1, const double* f2, int64_t n,
                                                    double* partial) {
    __shared__ double red[3][256];
    double s0 = 0., s1 = 0., s2 = 0.;
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        s0 += f0[i]; s1 += f1[i]; s2 += f2[i];
    }
    red[0][threadIdx.x] = s0; red[1][threadIdx.x] = s1; red[2][threadIdx.x] = s2;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (static_cast<int>(threadIdx.x) < w) {
            red[0][threadIdx.x] += red[0][threadIdx.x + w];
            red[1][threadIdx.x] += red[1][threadIdx.x + w];
            red[2][threadIdx.x] += red[2][threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partial[3 * blockIdx.x + 0] = red[0][0];
        partial[3 * blockIdx.x + 1] = red[1][0];
        partial[3 * blockIdx.x + 2] = red[2][0];
    }
}

}  // namespace

// 32-bit element offsets when every cell array holds fewer than 2^28 doubles.
bool narrow(int64_t n) { return n < (int64_t{1} << 28); }

hipError_t launch_mag_stage(const StageArgs& a, int64_t n, hipStream_t s, const uint32_t* ids, int64_t count) {
    if (ids) {
        const dim3 grid(static_cast<unsigned>((count + 255) / 256));
        const auto list = a.mixed ? mag_stage_list_kernel<uint32_t, true> : mag_stage_list_kernel<uint32_t, false>;
        if (count > 0 && narrow(n))
            hipLaunchKernelGGL(list, grid, dim3(256), 0, s, a, ids, static_cast<uint32_t>(count));
        else if (count > 0)
            hipLaunchKernelGGL((mag_stage_list_kernel<int64_t, true>), grid, dim3(256), 0, s, a, ids, count);
        return hipGetLastError();
    }
    const int64_t blocks = (n + 255) / 256;
    const auto stage = !narrow(n)  ? mag_stage_kernel<int64_t, true>
                       : a.mixed ? mag_stage_kernel<uint32_t, true>
                                 : mag_stage_kernel<uint32_t, false>;
    hipLaunchKernelGGL(stage, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_mag_stage_fused(const StageArgs& a, const FusedZArgs& f, bool hspec, hipStream_t s) {
    const int nz = static_cast<int>(a.nz);
    const int pairs = f.P > 1 ? f.P / 2 : 1;
    const bool lean = !a.rotate && !a.strain[0] && !a.hnu[0] && !a.hdrive[0] && !a.hcell[0] && !a.dm_out[0] &&
                      !a.prescribe && a.nmat >= 1 && a.nmat <= kLeanMats;
    const size_t lds = sizeof(double2) * (nz / 2 + fft_lds_elems(3 * pairs * nz)) +
                       (lean ? sizeof(DevMaterial) * static_cast<size_t>(a.nmat) : 0);
    const unsigned groups = static_cast<unsigned>(a.nx * a.ny / f.P);
    const bool n32 = narrow(a.nx * a.ny * a.nz);
    const dim3 g(groups), t(256);
    auto stage = mag_stage_fused_kernel<false, false, true, int64_t>;
    if (n32 && a.mixed)
        stage = !hspec ? mag_stage_fused_kernel<false, false, true, uint32_t>
                : lean ? mag_stage_fused_kernel<true, true, true, uint32_t>
                       : mag_stage_fused_kernel<true, false, true, uint32_t>;
    else if (n32)
        stage = !hspec ? mag_stage_fused_kernel<false, false, false, uint32_t>
                : lean ? mag_stage_fused_kernel<true, true, false, uint32_t>
                       : mag_stage_fused_kernel<true, false, false, uint32_t>;
    else if (hspec)
        stage = lean ? mag_stage_fused_kernel<true, true, true, int64_t> : mag_stage_fused_kernel<true, false, true, int64_t>;
    hipLaunchKernelGGL(stage, g, t, lds, s, a, f);
    return hipGetLastError();
}

hipError_t launch_afm_stage(const AfmStageArgs& a, int64_t n, hipStream_t s) {
    const int64_t blocks = (n + 255) / 256;
    const dim3 grid(static_cast<unsigned>((blocks + 7) / 8 * 16));
    const auto stage = !narrow(n)  ? afm_stage_kernel<int64_t, true>
                       : a.mixed ? afm_stage_kernel<uint32_t, true>
                                 : afm_stage_kernel<uint32_t, false>;
    hipLaunchKernelGGL(stage, grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_mag_batch(const StageArgs* items, const BatchLaunch& L, int stage, hipStream_t s) {
    const auto batch = !L.narrow ? mag_batch_kernel<int64_t, true>
                       : L.mixed ? mag_batch_kernel<uint32_t, true>
                                 : mag_batch_kernel<uint32_t, false>;
    hipLaunchKernelGGL(batch, dim3(L.grid), dim3(L.threads), 0, s, items, L, stage);
    return hipGetLastError();
}

hipError_t launch_afm_batch(const AfmStageArgs* items, const BatchLaunch& L, int stage, hipStream_t s) {
    // L.grid counts slots; the grid covers both sublattices of each
    const unsigned grid = 2u * ((L.grid + 7u) / 8u * 8u);
    const bool one = L.cpt == 1 && L.grid == L.total;
    auto batch = one ? afm_batch_kernel<int64_t, true, true> : afm_batch_kernel<int64_t, false, true>;
    if (L.narrow && L.mixed)
        batch = one ? afm_batch_kernel<uint32_t, true, true> : afm_batch_kernel<uint32_t, false, true>;
    else if (L.narrow)
        batch = one ? afm_batch_kernel<uint32_t, true, false> : afm_batch_kernel<uint32_t, false, false>;
    hipLaunchKernelGGL(batch, dim3(grid), dim3(L.threads), 0, s, items, L, stage);
    return hipGetLastError();
}

hipError_t launch_batch_clock(BatchClock* clk, StageArgs* fm, AfmStageArgs* afm, int count, hipStream_t s) {
    hipLaunchKernelGGL(batch_clock_kernel, dim3(static_cast<unsigned>((count + 255) / 256)), dim3(256), 0, s, clk, fm,
                       afm, count);
    return hipGetLastError();
}

hipError_t launch_prescribe_plane(double* const* m, const uint32_t* code, int64_t nx, int64_t ny, int64_t nz,
                                  const double v[3], hipStream_t s) {
    const int64_t nxy = nx * ny;
    hipLaunchKernelGGL(prescribe_plane_kernel, dim3(static_cast<unsigned>((nxy + 255) / 256)), dim3(256), 0, s,
                       m[0], m[1], m[2], code, nxy, nz, v[0], v[1], v[2]);
    return hipGetLastError();
}

hipError_t launch_sum3(const double* const* f, int64_t n, double* partial, int64_t blocks, hipStream_t s) {
    hipLaunchKernelGGL(sum3_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, f[0], f[1], f[2], n,
                       partial);
    return hipGetLastError();
}

}  // namespace gf
