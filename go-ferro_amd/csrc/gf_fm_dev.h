// gf_fm_dev.h — one ferromagnetic cell of an RK4 stage: its loads, effective
// field, LLG increment and update.  Shared by the magnet launches
// (gf_llg.hip) and the launch that runs a magnet stage beside the elastic
// force (gf_elastic.hip).
#pragma once

#include "gf_llg_dev.h"

namespace gf {

namespace {

// gather6 for launches whose active lanes hold consecutive cells along z
// (lane i of a wave at cell id0 + i, and a lane without a cell only past
// the grid's last cell): a cell's z neighbours are then the store values
// of the lanes next to it, moved with DPP wave shifts, except at a column
// end (k = 0 or nz - 1, where the neighbour wraps or the face is a surface)
// or a wave edge, where they are loaded.  A lane next to one without a cell
// is at a column end.  Two parts: the loads, and after the cell's other
// loads have been issued, the lane shifts of its own store c.
template <bool kMixed, class I>
__device__ __forceinline__ void gather6_lanes_load(const P3 s3, const uint32_t* code, I x, I y, I z, I nx, I ny, I nz,
                                                   double (&v)[6][3], uint32_t (&cd)[6]) {
    auto face = [&](int f) {
        const I nb = face_nb<I>(f, x, y, z, nx, ny, nz);
        for (int q = 0; q < 3; q++) v[f][q] = ldd(s3.p[q], nb);
        if (kMixed) cd[f] = ldu(code, nb);
    };
#pragma unroll
    for (int f = 0; f < 4; f++) face(f);
    const int lane = static_cast<int>(threadIdx.x & 63u);
    if (lane == 0 || z == 0) face(4);
    if (lane == 63 || z == nz - 1) face(5);
}

template <bool kMixed, class I>
__device__ __forceinline__ void gather6_lanes_shift(I z, I nz, const double (&c)[3], uint32_t own, double (&v)[6][3],
                                                    uint32_t (&cd)[6]) {
    const int lane = static_cast<int>(threadIdx.x & 63u);
    const bool gm = lane == 0 || z == 0, gp = lane == 63 || z == nz - 1;
    for (int q = 0; q < 3; q++) {
        const double dn = lane_up(c[q]), up = lane_down(c[q]);
        if (!gm) v[4][q] = dn;
        if (!gp) v[5][q] = up;
    }
    if (kMixed) {
        const uint32_t dn = lane_up(own), up = lane_down(own);
        if (!gm) cd[4] = dn;
        if (!gp) cd[5] = up;
    }
}

// Every global input of one FM cell of a stage except the static field:
// loaded together, before the cell's own code is known, so that one
// memory round trip feeds the cell (all indices are in bounds whatever the
// code says).
struct FmIn {
    uint32_t own;
    double c[3];        // stage store at the cell
    double v[6][3];     // stage store at the six face neighbours (gather6)
    uint32_t cd[6];     // their codes, where they are read
    double m[3];        // m at the start of the step
    double acc[3];      // RK accumulator (read at stages 2-4)
};

// kLanes: the launch's lanes hold consecutive cells (see gather6_lanes).
template <class I, bool kLanes, bool kMixed>
__device__ __forceinline__ void fm_load(const StageArgs& a, I id, I x, I y, I z, FmIn& in) {
    in.own = ldu(a.code, id);
    const P3 sp = {{a.store[0], a.store[1], a.store[2]}};
    for (int c = 0; c < 3; c++) in.c[c] = ldd(a.store[c], id);
    const I nx = static_cast<I>(a.nx), ny = static_cast<I>(a.ny), nz = static_cast<I>(a.nz);
    if (kLanes) gather6_lanes_load<kMixed, I>(sp, a.code, x, y, z, nx, ny, nz, in.v, in.cd);
    else gather6<kMixed, I>(sp, a.code, x, y, z, nx, ny, nz, in.v, in.cd);
    // at stage 1 the stage store is m itself: read it once
    const bool same = a.base[0] == a.store[0] && a.base[1] == a.store[1] && a.base[2] == a.store[2];
    for (int c = 0; c < 3; c++) in.m[c] = same ? in.c[c] : ldd_nt(a.base[c], id);
    for (int c = 0; c < 3; c++) in.acc[c] = a.stage > 1 ? ldd_nt(a.acc[c], id) : 0.;
    if (kLanes) gather6_lanes_shift<kMixed, I>(z, nz, in.c, in.own, in.v, in.cd);
}

// RK update of one component (see the file comment) from its preloaded m
// and accumulator; returns the value written to the next store (m itself
// at stage 4): the RK value, or pv where the cell's value is prescribed.
template <class I>
__device__ __forceinline__ double rk_store(int stage, I id, int c, double k, double m, double acc,
                                           double* const* accp, double* const* out, bool prescribed = false,
                                           double pv = 0.) {
    double v;
    if (stage == 1) {
        v = m + k * 0.5;
        std_nt(accp[c], id, k * kSixth);
    } else if (stage == 2) {
        v = m + k * 0.5;
        std_nt(accp[c], id, acc + k * kThird);
    } else if (stage == 3) {
        v = m + k;
        std_nt(accp[c], id, acc + k * kThird);
    } else {
        v = m + (acc + k * kSixth);
    }
    if (prescribed) v = pv;
    std_nt(out[c], id, v);
    return v;
}

// One FM cell of a stage: H_eff with the static field hs, the LLG
// increment and the RK update; n receives the next store value.  kLean
// compiles out the frame rotation and the optional fields (strain, non-
// uniform and shaped drives, electrodynamic back-action, k output, the
// prescribed bottom layer) for contexts that have none of them: their
// pointers and the rotation matrices then occupy no scalar registers
// across the cell loop.  mats is the material table, in global memory
// (GMat) or a workgroup's LDS copy (LMat).  z is the cell's.
template <bool kLean, bool kMixed, class I, class MT>
__device__ __forceinline__ void fm_cell(const StageArgs& a, MT* mats, const FmIn& in, I id, I z, double hs0, double hs1,
                                        double hs2, double& n0, double& n1, double& n2) {
    MT& M = mats[(in.own & kMatMask) - 1];

    const double mgx = in.c[0], mgy = in.c[1], mgz = in.c[2];
    double mx = mgx, my = mgy, mz = mgz;
    if (!kLean && a.rotate) rot(a.Tg2c, mgx, mgy, mgz, mx, my, mz);

    const Stencil st = magnet_stencil<true, kMixed>(in.c, in.v, in.cd, mats, in.own, kFmSurfShift, -1, a.idx, a.idy,
                                                    a.idz, M.Aex, M.Aex_self, M.dmi_slope);

    // magnetocrystalline anisotropy (magnetic_solver.cpp:124-141)
    double hac0 = 0., hac1 = 0., hac2 = 0.;
    if (M.anis_type == 1) {
        hac0 = -2. * (M.K1n * (my * my + mz * mz) + M.K2n * my * my * mz * mz) * mx;
        hac1 = -2. * (M.K1n * (mx * mx + mz * mz) + M.K2n * mx * mx * mz * mz) * my;
        hac2 = -2. * (M.K1n * (mx * mx + my * my) + M.K2n * mx * mx * my * my) * mz;
    } else if (M.anis_type == 2) {
        hac2 = 2. * M.K1n * mz;
    }
    double ha0 = hac0, ha1 = hac1, ha2 = hac2;
    if (!kLean && a.rotate) rot(a.Tc2g, hac0, hac1, hac2, ha0, ha1, ha2);

    // H_eff (magnetic_solver.cpp:164-198); the magnetoelastic term
    // (:89-96, 143-150) enters only when a strain is coupled, since it is
    // zero otherwise.
    double H0 = hs0 + ha0;
    double H1 = hs1 + ha1;
    double H2 = hs2 + ha2;
    if (!kLean && a.strain[0]) {
        double he0, he1, he2;
        magnetoelastic(a.strain, a.strain0, id, -2., M.B1n, M.B2n, mx, my, mz, a.rotate, a.Tc2g, he0, he1, he2);
        H0 = H0 + he0;
        H1 = H1 + he1;
        H2 = H2 + he2;
    }
    H0 = H0 + M.exch * st.ex[0] + M.dmi_pos * st.d[2] + a.hext[0];
    H1 = H1 + M.exch * st.ex[1] + M.dmi_pos * st.d[3] + a.hext[1];
    H2 = H2 + M.exch * st.ex[2] + M.dmi_neg * (st.d[0] + st.d[1]) + a.hext[2];
    if (!kLean && a.hnu[0]) {
        H0 = H0 + ldd(a.hnu[0], id);
        H1 = H1 + ldd(a.hnu[1], id);
        H2 = H2 + ldd(a.hnu[2], id);
    }
    if (!kLean && a.hdrive[0]) {
        H0 = H0 + ldd(a.hdrive[0], id) * a.drive_s;
        H1 = H1 + ldd(a.hdrive[1], id) * a.drive_s;
        H2 = H2 + ldd(a.hdrive[2], id) * a.drive_s;
    }
    if (!kLean && a.hcell[0]) {
        // electrodynamic back-action (magnetic_solver.cpp:200-204)
        H0 = H0 + ldd(a.hcell[0], id);
        H1 = H1 + ldd(a.hcell[1], id);
        H2 = H2 + ldd(a.hcell[2], id);
    }

    // LLG right-hand side times dt (magnetic_solver.cpp:206-220)
    const double px = mgy * H2 - mgz * H1, py = mgz * H0 - mgx * H2, pz = mgx * H1 - mgy * H0;
    const double qx = mgy * pz - mgz * py, qy = mgz * px - mgx * pz, qz = mgx * py - mgy * px;
    const double k0 = M.precess * px + M.alpha_precess * qx;
    const double k1 = M.precess * py + M.alpha_precess * qy;
    const double k2 = M.precess * pz + M.alpha_precess * qz;
    if (!kLean && a.dm_out[0]) {
        std_(a.dm_out[0], id, k0); std_(a.dm_out[1], id, k1); std_(a.dm_out[2], id, k2);
    }
    // update_prescribed_m{_half,_full,} over the update (magnetic_solver.cpp:
    // 1526-1609, 1891-1957); the accumulator keeps the LLG increment
    const bool pres = !kLean && a.prescribe && z == 0;
    n0 = rk_store(a.stage, id, 0, k0, in.m[0], in.acc[0], a.acc, a.out, pres, a.presc_m[0]);
    n1 = rk_store(a.stage, id, 1, k1, in.m[1], in.acc[1], a.acc, a.out, pres, a.presc_m[1]);
    n2 = rk_store(a.stage, id, 2, k2, in.m[2], in.acc[2], a.acc, a.out, pres, a.presc_m[2]);
}

// One FM cell of the unfused stage: coordinates from the linear index,
// magnetostatic field from Hstat.
template <class I, bool kLanes, bool kMixed>
__device__ __forceinline__ void fm_point(const StageArgs& a, I id) {
    const I ny = static_cast<I>(a.ny), nz = static_cast<I>(a.nz);
    I x, y, z;
    cell_xyz(a.div, id, ny, nz, x, y, z);
    FmIn in;
    fm_load<I, kLanes, kMixed>(a, id, x, y, z, in);
    // a null Hstat is zero (no statics, nothing uploaded)
    const bool hs = a.hstat[0] != nullptr;
    const double hs0 = hs ? ldd(a.hstat[0], id) : 0., hs1 = hs ? ldd(a.hstat[1], id) : 0.;
    const double hs2 = hs ? ldd(a.hstat[2], id) : 0.;
    if (!(in.own & kIsFM)) return;
    double n0, n1, n2;
    fm_cell<false, kMixed, I>(a, (GMat*)a.mats, in, id, z, hs0, hs1, hs2, n0, n1, n2);
}

}  // namespace

}  // namespace gf
