// gf_em_dev.h — device code of the electrodynamics stage shared by the EM
// launches and the launch that runs a ferroelectric stage beside them.
// Ampere per edge with the four-cell means of permittivity, conductivity,
// Jf, Jp and dp (get_dE_RK*, EMdynamic_solver.cpp:337-2237) fused with the
// RK update (update_DE_RK*, :3588-3777); Faraday per face with dM of the two
// cells (get_dH_RK*, :2239-3475) fused with update_DH_RK* (:3477-3586).
// RK4 keeps a state accumulator, acc = y + k1/6, acc += k2/3, acc += k3/3,
// y = acc + k4/6, the reference's left-to-right sum.
// On a thin column (8x8x1024: 65k cells, 230k edges, 200k faces) a launch is
// a few waves per SIMD, so the depth of the chain of loads and the index
// arithmetic (64-bit divisions) set its time: all reads of an edge or face
// go out together and offsets are 32-bit where they reach.  The launch with the
// ferroelectric cells took 13.8 us, 12.8 with that, 11.6 once it held the z walls
// and the cells' E too, and 10.0 to 10.6 since the components of an edge's and a
// face's reads are constants, so that the arrays' bases stay scalar.  On millions
// of cells bandwidth sets it, and no array is read that the stage does not use:
// 128x128x128 with a magnet 1053 us a step before the reads were grouped, 959 now.
#pragma once

#include "gf_llg_dev.h"

namespace gf {
namespace em_dev {

// Edges and faces of an EM grid: the elements of the E and of the H arrays.
__host__ __device__ __forceinline__ int64_t em_edges(const EmArgs& a) {
    return a.nx * (a.ny + 1) * (a.nz + 1) + (a.nx + 1) * a.ny * (a.nz + 1) + (a.nx + 1) * (a.ny + 1) * a.nz;
}
__host__ __device__ __forceinline__ int64_t em_faces(const EmArgs& a) {
    return (a.nx + 1) * a.ny * a.nz + a.nx * (a.ny + 1) * a.nz + a.nx * a.ny * (a.nz + 1);
}

// Workgroups of kEmGroup threads: those of the edges come first, then those
// of the faces, each kind rounded up (a workgroup has one kind only).
constexpr int kEmGroup = 256;
__host__ __device__ __forceinline__ unsigned em_groups(int64_t n) {
    return static_cast<unsigned>((n + kEmGroup - 1) / kEmGroup);
}

// RK update of element i from its preloaded base (at stages 1-3) and (at
// stages 2-4) accumulator.
template <class I>
__device__ __forceinline__ void rk_state(int stage, I i, double k, double y, double ac, double* base, double* acc,
                                         double* out) {
    if (stage == 1) {
        std_(out, i, y + k * 0.5);
        std_(acc, i, y + k * kSixth);
    } else if (stage == 2) {
        std_(out, i, y + k * 0.5);
        std_(acc, i, ac + k * kThird);
    } else if (stage == 3) {
        std_(out, i, y + k);
        std_(acc, i, ac + k * kThird);
    } else {
        std_(base, i, ac + k * kSixth);
    }
}

// The workgroup's LDS copy of what an edge needs of every material: the
// relative permittivity, the conductivity and whether it is ferroelectric.
// An edge waits for its cells' codes and then for an LDS read, not for a
// second trip to global memory.
constexpr int kEmC = 3;

__device__ __forceinline__ void load_emtab(double* tab, const DevMaterial* mats, int nmat) {
    for (int t = threadIdx.x; t < kEmC * nmat; t += blockDim.x) {
        const DevMaterial& M = mats[t / kEmC];
        const int q = t % kEmC;
        tab[t] = q == 0 ? M.em_er : q == 1 ? M.em_cond : (M.is_fe ? 1. : 0.);
    }
    __syncthreads();
}

// The free current of cell (i, j, k), component comp, at the stage time:
// the value update_Jf_input* writes in its box (EMdynamic_solver.cpp:
// 3885-4315), zero elsewhere.
__device__ __forceinline__ double jf_at(const EmArgs& a, int comp, int64_t i, int64_t j, int64_t k) {
    if (comp != a.jf_comp || i < a.jf_lo[0] || i > a.jf_hi[0] || j < a.jf_lo[1] || j > a.jf_hi[1] || k < a.jf_lo[2] ||
        k > a.jf_hi[2])
        return 0.;
    return a.jf_spatial ? a.jf_value * a.jf_spatial[k - a.jf_lo[2]] : a.jf_value;
}

// Four-cell means around an edge and the Ampere increment
// (EMdynamic_solver.cpp:392-499), with the spin-pumping current on x and y.
// The cells are (ci, cj, ck)[q], index cell[q], codes tq[q], q store qv[q];
// the quotients by four, the cell count and dt are products with their
// reciprocals (within an ulp of the reference's).
template <class I>
__device__ __forceinline__ double edge_increment(const EmArgs& a, const double* tab, int comp, const I (&cell)[4],
                                                 const I (&ci)[4], const I (&cj)[4], const I (&ck)[4],
                                                 const uint32_t (&tq)[4], const double (&qv)[4], double curl,
                                                 double e_store) {
    double Jf = 0., Jp = 0., Ji = 0., dP = 0., er = 0., cond = 0., pc = 0.;
    for (int q = 0; q < 4; q++) {
        const I id = cell[q];
        const uint32_t t = tq[q] & kMatMask;
        if (!t) {
            er = er + 1.;
        } else {
            const double* M = tab + (t - 1u) * kEmC;
            dP = dP + qv[q] * a.dt;
            er = er + M[0];
            cond = cond + M[1];
            pc = pc + M[2];
        }
        if (a.jf_comp >= 0) Jf = Jf + jf_at(a, comp, ci[q], cj[q], ck[q]);
        if (a.jps[0]) Jp = Jp + ldd(a.jps[comp], id) + ldd(a.jps[3 + comp], id) + ldd(a.jps[6 + comp], id);
        if (a.jishe[0] && comp < 2) Ji = Ji + ldd(a.jishe[comp], id);
    }
    const double rpc = pc < 1.5 ? 1. : (pc < 2.5 ? 0.5 : (pc < 3.5 ? kThird : 0.25));
    Jf = Jf * 0.25;
    Jp = Jp * 0.25;
    Ji = Ji * 0.25;
    dP = dP * rpc;
    er = er * 0.25;
    cond = cond * 0.25;
    return a.ce / er * (curl - Jf - Jp - Ji - cond * e_store - dP * a.rdt);
}

// The new value of the wall edge e of a z wall (top: k = nz) from its base yw,
// the base y and the new value yn of the edge next to it, in: the first-order
// Mur condition, or zero (EMdynamic_AbsorbingBoundary.cpp:58-874).  At stage 4
// the bases are those kept at stage 3, since the edges overwrite theirs.
template <class I>
__device__ __forceinline__ double z_wall_edge(const EmArgs& a, int comp, bool top, I e, I in, double yw, double y,
                                              double yn) {
    if (a.wall_zero[top]) return 0.;
    if (a.stage < 4) return y + a.wall_cf[top] * (yw - yn);
    return ldd(a.t1[comp], in) + a.wall_cf[top] * (ldd(a.t1[comp], e) - yn);
}

// Ampere on edge e of the concatenated Ex|Ey|Ez grids, with its RK update.
// Everything an edge reads (its base, accumulator and store, the H store
// around it, its cells' codes and q store) is loaded before any of it is
// used: every index is in bounds, on the wall edges too (they wrap).
// A whole workgroup calls it, with e past the last edge in the last one's
// spare threads: tab is the workgroup's material table, staged here after
// the edge's own loads have been issued, so that both take one round trip.
template <class I, bool kQ, bool kWall>
__device__ __forceinline__ void em_edge(const EmArgs& a, double* tab, I e) {
    const I nE = static_cast<I>(em_edges(a));
    const bool live = e < nE;
    if (!live) e = nE - 1;
    const I nx = static_cast<I>(a.nx), ny = static_cast<I>(a.ny), nz = static_cast<I>(a.nz);
    const I nEx = nx * (ny + 1) * (nz + 1), nEy = (nx + 1) * ny * (nz + 1);
    auto C = [&](I i, I j, I k) { return (i * ny + j) * nz + k; };
    auto HY = [&](I i, I j, I k) { return (i * (ny + 1) + j) * nz + k; };
    auto HZ = [&](I i, I j, I k) { return (i * ny + j) * (nz + 1) + k; };
    auto near = [](I v, I n) { return v <= 1 || v >= n - 1; };
    const bool last = a.stage == 4;
    int comp, wall = 0;   // -1, 1: an edge of the bottom, top z wall whose thread takes the one next to it first
    bool hist, dead;      // on a plane a Mur wall reads (two next to each non-periodic wall); a wall edge
    I in;                 // the edge whose increment this thread evaluates
    I cell[4], ci[4], cj[4], ck[4], hp[4];
    uint32_t tq[4];
    double y, yw, ac, es, rh[2], hv[4], qv[4] = {0., 0., 0., 0.};
    // The reads of an edge of component c, whose curl is (H_h0[hp0] - H_h0[hp1])
    // rh0 - (H_h1[hp2] - H_h1[hp3]) rh1; c, h0 and h1 are constants of each
    // call, so that the arrays' bases stay in scalar registers.
    auto read = [&](int c, int h0, int h1) __attribute__((always_inline)) {
        comp = c;
        // A wall's thread reads what its neighbour's own thread may write in
        // this launch only at the stages where it does not (the base before
        // stage 4, the accumulator at stage 4).
        in = wall == 0 ? e : (wall < 0 ? e + 1 : e - 1);
        // at stage 4 the base is read only to keep it (a whole array less to read)
        y = !last || (a.keep && hist && !wall) ? ldd(a.eb[c], in) : 0.;
        yw = wall && !last ? ldd(a.eb[c], e) : 0.;
        ac = (wall ? last : a.stage > 1) ? ldd(a.eacc[c], in) : 0.;
        es = ldd(a.es[c], in);
        for (int q = 0; q < 4; q++) {
            cell[q] = C(ci[q], cj[q], ck[q]);
            tq[q] = ldu(a.code, cell[q]);
            hv[q] = ldd(a.hs[q < 2 ? h0 : h1], hp[q]);
            if (kQ && a.q[0]) qv[q] = ldd(a.q[c], cell[q]);
        }
    };
    if (e < nEx) {
        const I l = e / (nz + 1), i = l / (ny + 1), j = l - i * (ny + 1);
        I k = e - l * (nz + 1);
        hist = (!a.per[1] && near(j, ny)) || (!a.per[2] && near(k, nz));
        if (kWall && a.zwall && (k == 0 || k == nz)) { wall = k == 0 ? -1 : 1; k = k == 0 ? 1 : nz - 1; }
        const bool wj = j == 0 || j == ny, wk = k == 0 || k == nz;
        dead = (wj && !a.per[1]) || (wk && !a.per[2]);
        const I y1 = wj ? ny - 1 : j - 1, y3 = wj ? 0 : j, z1 = wk ? nz - 1 : k - 1, z2 = wk ? 0 : k;
        for (int q = 0; q < 4; q++) { ci[q] = i; cj[q] = q < 2 ? y1 : y3; ck[q] = q & 1 ? z2 : z1; }
        rh[0] = a.rdy; rh[1] = a.rdz;
        hp[0] = HZ(i, y3, z2); hp[1] = HZ(i, y1, z2); hp[2] = HY(i, y3, z2); hp[3] = HY(i, y3, z1);
        read(0, 2, 1);
    } else if (e < nEx + nEy) {
        e -= nEx;
        const I l = e / (nz + 1), i = l / ny, j = l - i * ny;
        I k = e - l * (nz + 1);
        hist = (!a.per[0] && near(i, nx)) || (!a.per[2] && near(k, nz));
        if (kWall && a.zwall && (k == 0 || k == nz)) { wall = k == 0 ? -1 : 1; k = k == 0 ? 1 : nz - 1; }
        const bool wi = i == 0 || i == nx, wk = k == 0 || k == nz;
        dead = (wi && !a.per[0]) || (wk && !a.per[2]);
        const I x1 = wi ? nx - 1 : i - 1, x3 = wi ? 0 : i, z1 = wk ? nz - 1 : k - 1, z2 = wk ? 0 : k;
        for (int q = 0; q < 4; q++) { ci[q] = q < 2 ? x1 : x3; cj[q] = j; ck[q] = q & 1 ? z2 : z1; }
        rh[0] = a.rdz; rh[1] = a.rdx;
        hp[0] = C(x3, j, z2); hp[1] = C(x3, j, z1); hp[2] = HZ(x3, j, z2); hp[3] = HZ(x1, j, z2);
        read(1, 0, 2);
    } else {
        e -= nEx + nEy;
        const I l = e / nz, k = e - l * nz, i = l / (ny + 1), j = l - i * (ny + 1);
        hist = (!a.per[0] && near(i, nx)) || (!a.per[1] && near(j, ny));
        const bool wi = i == 0 || i == nx, wj = j == 0 || j == ny;
        dead = (wi && !a.per[0]) || (wj && !a.per[1]);
        const I x1 = wi ? nx - 1 : i - 1, x3 = wi ? 0 : i, y1 = wj ? ny - 1 : j - 1, y2 = wj ? 0 : j;
        for (int q = 0; q < 4; q++) { ci[q] = q < 2 ? x1 : x3; cj[q] = q & 1 ? y2 : y1; ck[q] = k; }
        rh[0] = a.rdx; rh[1] = a.rdy;
        hp[0] = HY(x3, y2, k); hp[1] = HY(x1, y2, k); hp[2] = C(x3, y2, k); hp[3] = C(x3, y1, k);
        read(2, 1, 0);
    }
    load_emtab(tab, a.mats, a.nmat);
    if (!live) return;
    double k_ = 0.;
    if (!dead)
        k_ = edge_increment<I>(a, tab, comp, cell, ci, cj, ck, tq, qv, (hv[0] - hv[1]) * rh[0] - (hv[2] - hv[3]) * rh[1],
                               es);
    if (wall) {
        const double yn = last ? ac + k_ * kSixth : y + (a.stage == 3 ? k_ : k_ * 0.5);
        std_(last ? a.eb[comp] : a.eo[comp], e, z_wall_edge<I>(a, comp, wall > 0, e, in, yw, y, yn));
        if (a.stage == 1) std_(a.eacc[comp], e, yw);
        if (a.keep) std_(a.t1[comp], e, yw);
        return;
    }
    // the base value before the combine overwrites it, for the Mur walls
    // (transfer_pointer, EMdynamic_AbsorbingBoundary.cpp:3-56); each edge's
    // own thread reads and then writes its base
    if (a.keep && hist) std_(a.t1[comp], e, y);
    rk_state<I>(a.stage, e, k_, y, ac, a.eb[comp], a.eacc[comp], a.eo[comp]);
}

// What dM of one cell next to a face takes (EMdynamic_solver.cpp:2290-2340),
// read only where a magnetic increment is given.
struct CellDm {
    uint32_t mat;
    double f, f1, f2;
};
template <class I>
__device__ __forceinline__ CellDm load_dm(const EmArgs& a, int comp, I id) {
    return {ldu(a.code, id) & kMatMask, a.dm[0] ? ldd(a.dm[comp], id) : 0., a.dma1[0] ? ldd(a.dma1[comp], id) : 0.,
            a.dma2[0] ? ldd(a.dma2[comp], id) : 0.};
}
__device__ __forceinline__ double cell_dm(const EmArgs& a, const CellDm& c, double& count) {
    if (!c.mat) return 0.;
    const DevMaterial& M = a.mats[c.mat - 1];
    if (M.is_fm || M.is_afm) count = count + 1.;
    return c.f * M.Ms + c.f1 * M.aMs[0] + c.f2 * M.aMs[1];
}

// Faraday on face f of the concatenated Hx|Hy|Hz grids, with its RK update;
// loads first, as em_edge.  Without magnetic increments the cells' part of
// the increment is zero and their codes are not read.
template <class I>
__device__ __forceinline__ void em_face(const EmArgs& a, I f) {
    const I nx = static_cast<I>(a.nx), ny = static_cast<I>(a.ny), nz = static_cast<I>(a.nz);
    const I nHx = (nx + 1) * ny * nz, nHy = nx * (ny + 1) * nz;
    auto C = [&](I i, I j, I k) { return (i * ny + j) * nz + k; };
    auto EX = [&](I i, I j, I k) { return (i * (ny + 1) + j) * (nz + 1) + k; };
    auto EY = [&](I i, I j, I k) { return (i * ny + j) * (nz + 1) + k; };
    auto EZ = [&](I i, I j, I k) { return (i * (ny + 1) + j) * nz + k; };
    const bool mag = a.dm[0] || a.dma1[0];
    int comp;
    CellDm m1{}, m2{};    // of the two cells beside the face
    double y, ac, re[2], ev[4];   // curl = (ev0 - ev1) re0 - (ev2 - ev3) re1
    // the cells first (their materials' records are a second trip to memory),
    // with a constant component in each call
    auto read = [&](int c, I c1, I c2) __attribute__((always_inline)) {
        comp = c;
        if (mag) { m1 = load_dm<I>(a, c, c1); m2 = load_dm<I>(a, c, c2); }
        y = a.stage < 4 ? ldd(a.hb[c], f) : 0.;
        ac = a.stage > 1 ? ldd(a.hacc[c], f) : 0.;
    };
    if (f < nHx) {
        const I l = f / nz, k = f - l * nz, i = l / ny, j = l - i * ny;
        const I x1 = i == 0 ? (a.per[0] ? nx - 1 : 0) : i - 1, x2 = i == nx ? (a.per[0] ? 0 : nx - 1) : i;
        read(0, C(x1, j, k), C(x2, j, k));
        re[0] = a.rdy; re[1] = a.rdz;
        ev[0] = ldd(a.es[2], EZ(i, j + 1, k)); ev[1] = ldd(a.es[2], EZ(i, j, k));
        ev[2] = ldd(a.es[1] + 1, EY(i, j, k)); ev[3] = ldd(a.es[1], EY(i, j, k));
    } else if (f < nHx + nHy) {
        f -= nHx;
        const I l = f / nz, k = f - l * nz, i = l / (ny + 1), j = l - i * (ny + 1);
        const I y1 = j == 0 ? (a.per[1] ? ny - 1 : 0) : j - 1, y2 = j == ny ? (a.per[1] ? 0 : ny - 1) : j;
        read(1, C(i, y1, k), C(i, y2, k));
        re[0] = a.rdz; re[1] = a.rdx;
        ev[0] = ldd(a.es[0] + 1, EX(i, j, k)); ev[1] = ldd(a.es[0], EX(i, j, k));
        ev[2] = ldd(a.es[2], EZ(i + 1, j, k)); ev[3] = ldd(a.es[2], EZ(i, j, k));
    } else {
        f -= nHx + nHy;
        const I l = f / (nz + 1), k = f - l * (nz + 1), i = l / ny, j = l - i * ny;
        const I z1 = k == 0 ? (a.per[2] ? nz - 1 : 0) : k - 1, z2 = k == nz ? (a.per[2] ? 0 : nz - 1) : k;
        read(2, C(i, j, z1), C(i, j, z2));
        re[0] = a.rdx; re[1] = a.rdy;
        ev[0] = ldd(a.es[1], EY(i + 1, j, k)); ev[1] = ldd(a.es[1], EY(i, j, k));
        ev[2] = ldd(a.es[0], EX(i, j + 1, k)); ev[3] = ldd(a.es[0], EX(i, j, k));
    }
    double k_ = -a.dt / kMu0 * ((ev[0] - ev[1]) * re[0] - (ev[2] - ev[3]) * re[1]);
    if (mag) {
        double cnt = 0.;
        const double d1 = cell_dm(a, m1, cnt), d2 = cell_dm(a, m2, cnt);
        if (cnt < 0.5) cnt = 1.;
        k_ = k_ - (d1 + d2) / cnt;
    }
    rk_state<I>(a.stage, f, k_, y, ac, a.hb[comp], a.hacc[comp], a.ho[comp]);
}

}  // namespace em_dev
}  // namespace gf
