// gf_elastic.hip — elastodynamics RK4 stage for gfx950 (FP64).
//
// One stage of the reference's elastic solver (elastic_dynamic_solver.cpp,
// elastodynamics_AbsorbingBoundary.cpp) is two launches, with Mur planes three:
//   prep      face gradients of the u store and the cell strain (:107-227),
//             the eigenstrain from the m, m_AFM and p stores (:4-104) with
//             back-action, and each cell's part of its face stresses; at
//             stage 4 the boundary planes of u into the history ring
//             (transfer_pointer, elastodynamics_AbsorbingBoundary.cpp:3-89)
//   force     stress divergence, dv and du = v_s dt, the v and u RK updates
//             (get_dv_RKs / get_du_RKs / update_v_RKs / update_u_RKs, :841-3057),
//             the Liao plane and the displacement source
//             (elastodynamics_AbsorbingBoundary.cpp:92-230, :3060-3284)
//   boundary  Mur planes and the source: a Mur plane reads its neighbour's
//             new u, so it follows the update in a launch of its own
// The force launch reads the u store around each cell (its face gradients)
// and writes the next store into a second array (the two are swapped after
// it); v and its store are read and written by their own cell's thread only.
// The Liao plane k = 0 reads only the history, so the cell's own thread
// writes it, and the planes the history keeps are the prep's own cells: the
// two launches that did this took 4.2 and 2.7 us (70k cells) or 6.2 and 4.8 us
// (1M cells, of which the force gives 6 back).
//
// RK4 bookkeeping keeps a state accumulator per field, acc = y + k1/6,
// acc = acc + k2/3, acc = acc + k3/3, y = acc + k4/6, which is the
// reference's left-to-right y + k1/6 + k2/3 + k3/3 + k4/6 (the weights applied
// as products with the rounded reciprocals, within about an ulp of the quotients).
#include "gf_fm_dev.h"

namespace gf {

namespace {

__device__ __forceinline__ bool solid(const uint32_t* code, int64_t id) { return (code[id] & kMatMask) != 0u; }

__device__ __forceinline__ void rot_vec(const double T[3][3], double ix, double iy, double iz, double& ox,
                                        double& oy, double& oz) {
    ox = T[0][0] * ix + T[0][1] * iy + T[0][2] * iz;
    oy = T[1][0] * ix + T[1][1] * iy + T[1][2] * iz;
    oz = T[2][0] * ix + T[2][1] * iy + T[2][2] * iz;
}

// o_ij = sum_kl T_ik T_jl s_kl of a symmetric tensor given in Voigt order,
// result in Voigt order (mathlib.cpp:78-125, summed k-major as there).
__device__ __forceinline__ void rot_voigt(const double T[3][3], const double v[6], double o[6]) {
    const double s[3][3] = {{v[0], v[5], v[4]}, {v[5], v[1], v[3]}, {v[4], v[3], v[2]}};
    const int oi[6] = {0, 1, 2, 1, 0, 0};
    const int oj[6] = {0, 1, 2, 2, 2, 1};
    for (int c = 0; c < 6; c++) {
        const int i = oi[c], j = oj[c];
        double r = 0.;
        for (int k = 0; k < 3; k++)
            for (int l = 0; l < 3; l++) r = r + T[i][k] * T[j][l] * s[k][l];
        o[c] = r;
    }
}

// ---------------------------------------------------------------- strain
// (i, j, k) of cell id, with 32-bit arithmetic when the grid is narrow.
__device__ __forceinline__ void cell_ijk(const ElStrainArgs& a, int64_t id, int64_t& i, int64_t& j, int64_t& k) {
    if (a.nx * a.ny * a.nz < (int64_t{1} << 28)) {
        uint32_t x, y, z;
        cell_xyz(a.div, static_cast<uint32_t>(id), static_cast<uint32_t>(a.ny), static_cast<uint32_t>(a.nz), x, y, z);
        i = x; j = y; k = z;
    } else {
        cell_xyz(a.div, id, a.ny, a.nz, i, j, k);
    }
}

// Face gradients g[face][comp] of cell id = (i, j, k) of the u store,
// faces ordered x-, x+, y-, y+, z-, z+.  A stress-free face (vacuum on a
// side, or a non-periodic wall) has zero gradient; across a periodic wall
// the difference wraps (elastic_dynamic_solver.cpp:107-187).  The
// differences are multiplied by the reciprocal spacings (within an ulp of
// the reference's quotients); the upper face of a cell and the lower face
// of the cell above it are the same expression, hence the same value.
// The cell's face gradients from the u store.  Every load is issued before
// any code is known (all indices are in bounds), so that one memory round
// trip feeds the cell; the launches that call it run consecutive cells in
// consecutive lanes (one cell per thread, none past the grid's last cell),
// so the z neighbours' values and codes come from the adjacent lanes (DPP
// wave shifts) except at a column end or a wave edge, where they are
// loaded.
__device__ __forceinline__ void cell_grad(const ElStrainArgs& a, int64_t id, int64_t i, int64_t j, int64_t k,
                                          double (&g)[6][3]) {
    const int64_t nx = a.nx, ny = a.ny, nz = a.nz;
    const int64_t nb[6] = {((i == 0 ? nx - 1 : i - 1) * ny + j) * nz + k, ((i == nx - 1 ? 0 : i + 1) * ny + j) * nz + k,
                           (i * ny + (j == 0 ? ny - 1 : j - 1)) * nz + k, (i * ny + (j == ny - 1 ? 0 : j + 1)) * nz + k,
                           (i * ny + j) * nz + (k == 0 ? nz - 1 : k - 1), (i * ny + j) * nz + (k == nz - 1 ? 0 : k + 1)};
    const uint32_t own = a.code[id];
    double u[3], un[6][3];
    uint32_t cn[6];
    for (int c = 0; c < 3; c++) u[c] = a.us[c][id];
    for (int f = 0; f < 4; f++) {
        for (int c = 0; c < 3; c++) un[f][c] = a.us[c][nb[f]];
        cn[f] = a.code[nb[f]];
    }
    const int lane = static_cast<int>(threadIdx.x & 63u);
    const bool gm = lane == 0 || k == 0, gp = lane == 63 || k == nz - 1;
    if (gm) {
        for (int c = 0; c < 3; c++) un[4][c] = a.us[c][nb[4]];
        cn[4] = a.code[nb[4]];
    }
    if (gp) {
        for (int c = 0; c < 3; c++) un[5][c] = a.us[c][nb[5]];
        cn[5] = a.code[nb[5]];
    }
    for (int c = 0; c < 3; c++) {
        const double dn = lane_up(u[c]), up = lane_down(u[c]);
        if (!gm) un[4][c] = dn;
        if (!gp) un[5][c] = up;
    }
    const uint32_t cdn = lane_up(own), cup = lane_down(own);
    if (!gm) cn[4] = cdn;
    if (!gp) cn[5] = cup;
    const bool me = (own & kMatMask) != 0u;
    const bool wall[6] = {i == 0 && !a.per[0], i == nx - 1 && !a.per[0], j == 0 && !a.per[1],
                          j == ny - 1 && !a.per[1], k == 0 && !a.per[2], k == nz - 1 && !a.per[2]};
    const double ih[3] = {a.idx, a.idy, a.idz};
    for (int f = 0; f < 6; f++) {
        const bool fr = wall[f] || !(me && (cn[f] & kMatMask) != 0u);
        for (int c = 0; c < 3; c++) {
            if (fr) g[f][c] = 0.;
            else if (f & 1) g[f][c] = (un[f][c] - u[c]) * ih[f >> 1];
            else g[f][c] = (u[c] - un[f][c]) * ih[f >> 1];
        }
    }
}

// The face arrays: a cell writes its lower faces, the last cell along an
// axis its upper face too.
__device__ __forceinline__ void grad_out(const ElStrainArgs& a, int64_t i, int64_t j, int64_t k,
                                         const double (&g)[6][3]) {
    const int64_t nx = a.nx, ny = a.ny, nz = a.nz;
    for (int c = 0; c < 3; c++) {
        a.gyz[c][(i * ny + j) * nz + k] = g[0][c];
        if (i == nx - 1) a.gyz[c][(nx * ny + j) * nz + k] = g[1][c];
        a.gxz[c][(i * (ny + 1) + j) * nz + k] = g[2][c];
        if (j == ny - 1) a.gxz[c][(i * (ny + 1) + ny) * nz + k] = g[3][c];
        a.gxy[c][(i * ny + j) * (nz + 1) + k] = g[4][c];
        if (k == nz - 1) a.gxy[c][(i * ny + j) * (nz + 1) + nz] = g[5][c];
    }
}

// Cell strain as the average of its face gradients (:190-227).
__device__ __forceinline__ void strain_of(const double (&g)[6][3], double (&e)[6]) {
    e[0] = (g[0][0] + g[1][0]) / 2.;
    e[1] = (g[2][1] + g[3][1]) / 2.;
    e[2] = (g[4][2] + g[5][2]) / 2.;
    e[3] = (g[4][1] + g[5][1] + g[2][2] + g[3][2]) / 4.;
    e[4] = (g[4][0] + g[5][0] + g[0][2] + g[1][2]) / 4.;
    e[5] = (g[2][0] + g[3][0] + g[0][1] + g[1][1]) / 4.;
}

// The strain out, global frame and (rotated) crystal frame.
__device__ __forceinline__ void strain_out(const ElStrainArgs& a, int64_t id, const double (&e)[6]) {
    for (int c = 0; c < 6; c++) a.eg[c][id] = e[c];
    if (a.ec[0] != a.eg[0]) {
        double o[6];
        if (a.rotate) rot_voigt(a.Tg2c, e, o);
        else for (int c = 0; c < 6; c++) o[c] = e[c];
        for (int c = 0; c < 6; c++) a.ec[c][id] = o[c];
    }
}

__global__ void __launch_bounds__(256) el_strain_kernel(ElStrainArgs a) {
    const int64_t id = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (id >= a.nx * a.ny * a.nz) return;
    int64_t i, j, k;
    cell_ijk(a, id, i, j, k);
    double g[6][3], e[6];
    cell_grad(a, id, i, j, k, g);
    grad_out(a, i, j, k, g);
    strain_of(g, e);
    strain_out(a, id, e);
}

// ----------------------------------------------------------- eigenstrain
// Eigenstrain of cell id from the stage stores (elastic_dynamic_solver.cpp:
// 4-104) less the static eigenstrain at t0 when there is one: s in the
// crystal frame, o in the global frame, zero for vacuum.
// kGeneral: with rotation and the flexoelectric terms; the lean form is
// used only when the context has neither.  code is the cell's code; lc, when
// set, the workgroup's LDS copy of every material's constants (kEigC each:
// l100 l111 l100a l111a l100b l111b Q11 Q12 Q44).  The stores are read
// before the code is known (every index is in bounds), so one memory round
// trip feeds the cell.
constexpr int kEigC = 9;

template <bool kGeneral = true>
__device__ __forceinline__ void eigenstrain(const ElEigenArgs& a, const double* lc, int64_t id, uint32_t code,
                                            double s[6], double o[6]) {
    const uint32_t t = code & kMatMask;
    double v[4][3];
    const double* const* src[4] = {a.p, a.m, a.m1, a.m2};
    for (int f = 0; f < 4; f++) {
        v[f][0] = 0.; v[f][1] = 0.; v[f][2] = 0.;
        if (src[f][0]) { v[f][0] = src[f][0][id]; v[f][1] = src[f][1][id]; v[f][2] = src[f][2][id]; }
    }
    double t0[6] = {0., 0., 0., 0., 0., 0.};
    if (a.e0t0[0])
        for (int c = 0; c < 6; c++) t0[c] = a.e0t0[c][id];
    for (int c = 0; c < 6; c++) { s[c] = 0.; o[c] = 0.; }
    if (t) {
        double C[kEigC];
        if (lc) {
            for (int q = 0; q < kEigC; q++) C[q] = lc[(t - 1) * kEigC + q];
        } else {
            const DevMaterial& M = a.mats[t - 1];
            C[0] = M.l100; C[1] = M.l111; C[2] = M.l100a; C[3] = M.l111a; C[4] = M.l100b; C[5] = M.l111b;
            C[6] = M.Q11; C[7] = M.Q12; C[8] = M.Q44;
        }
        for (int f = 0; f < 4; f++) {
            const double x = v[f][0], y = v[f][1], z = v[f][2];
            if (kGeneral && a.rotate) rot_vec(a.Tg2c, x, y, z, v[f][0], v[f][1], v[f][2]);
        }
        const double px = v[0][0], py = v[0][1], pz = v[0][2];
        const double mx = v[1][0], my = v[1][1], mz = v[1][2];
        const double ax = v[2][0], ay = v[2][1], az = v[2][2];
        const double bx = v[3][0], by = v[3][1], bz = v[3][2];
        s[0] = 1.5 * C[0] * (mx * mx - 1. / 3.) + C[6] * (px * px) + C[7] * (py * py + pz * pz) +
               0.5 * 1.5 * C[2] * (ax * ax - 1. / 3.) + 0.5 * 1.5 * C[4] * (bx * bx - 1. / 3.) - t0[0];
        s[1] = 1.5 * C[0] * (my * my - 1. / 3.) + C[6] * (py * py) + C[7] * (px * px + pz * pz) +
               0.5 * 1.5 * C[2] * (ay * ay - 1. / 3.) + 0.5 * 1.5 * C[4] * (by * by - 1. / 3.) - t0[1];
        s[2] = 1.5 * C[0] * (mz * mz - 1. / 3.) + C[6] * (pz * pz) + C[7] * (py * py + px * px) +
               0.5 * 1.5 * C[2] * (az * az - 1. / 3.) + 0.5 * 1.5 * C[4] * (bz * bz - 1. / 3.) - t0[2];
        s[3] = 1.5 * C[1] * my * mz + C[8] * py * pz + 0.5 * 1.5 * C[3] * ay * az + 0.5 * 1.5 * C[5] * by * bz - t0[3];
        s[4] = 1.5 * C[1] * mx * mz + C[8] * px * pz + 0.5 * 1.5 * C[3] * ax * az + 0.5 * 1.5 * C[5] * bx * bz - t0[4];
        s[5] = 1.5 * C[1] * my * mx + C[8] * py * px + 0.5 * 1.5 * C[3] * ay * ax + 0.5 * 1.5 * C[5] * by * bx - t0[5];
        if (kGeneral && a.flexo) {
            // -F grad p (:82-89): the global-frame gradient of FE cells,
            // zero elsewhere, enters the crystal-frame tensor
            const FlexoMat& F = a.flexo[t - 1];
            double g[3][3] = {{0., 0., 0.}, {0., 0., 0.}, {0., 0., 0.}};
            const uint32_t own = a.code[id];
            if (own & kIsFE) {
                const int64_t nyz = a.ny * a.nz;
                const int64_t i = id / nyz, j = (id - i * nyz) / a.nz, k = id - i * nyz - j * a.nz;
                const double h[3] = {a.dx, a.dy, a.dz};
                fe_p_gradient(own, a.p, id, i, j, k, a.nx, a.ny, a.nz, h, g);
            }
            s[0] = s[0] - F.F11 * g[0][0] - F.F12 * (g[2][2] + g[1][1]);
            s[1] = s[1] - F.F11 * g[1][1] - F.F12 * (g[2][2] + g[0][0]);
            s[2] = s[2] - F.F11 * g[2][2] - F.F12 * (g[0][0] + g[1][1]);
            s[3] = s[3] - F.F44 / 2. * (g[1][2] + g[2][1]);
            s[4] = s[4] - F.F44 / 2. * (g[0][2] + g[2][0]);
            s[5] = s[5] - F.F44 / 2. * (g[1][0] + g[0][1]);
        }
        if (kGeneral && a.rotate) rot_voigt(a.Tc2g, s, o);
        else for (int c = 0; c < 6; c++) o[c] = s[c];
    }
}

// ----------------------------------------------------------------- force
__device__ __forceinline__ double crow(const double (*C)[6], int r, const double e[6]) {
    double s = 0.;
    for (int j = 0; j < 6; j++) s = s + C[r][j] * e[j];
    return s;
}

// The stress the reference evaluates on a face from the strain of one cell
// beside it is C e with (elastic_dynamic_solver.cpp:876-933, 994-1050,
// 1112-1166, 1229-1290)
//   YZ face (rows xx, xy, xz): e = [gx_f - e0xx, eyy - e0yy, ezz - e0zz,
//       2(eyz - e0yz), (gx_zb + gx_zt + 2 gz_f)/2 - 2 e0xz, (gx_yb + gx_yt + 2 gy_f)/2 - 2 e0xy]
//   XZ face (rows xy, yy, yz) and XY face (rows xz, yz, zz) likewise,
// where g?_f is the face's own gradient and the others belong to the cell
// (its strain e, eigenstrain e0, the gradients on its faces across the
// axis).  C e is linear in e, so it splits into a part of the cell, P =
// C (e with the face gradients zero), and C fp with fp holding the face
// gradients: the face gradient of component c of the face's axis a enters
// strain entry (a, c).  The face stress is the mean of its two cells'
// evaluations, (P_q + C_q fp + P_n + C_n fp) / 2: the prep launch writes
// P^x, P^y, P^z of every cell, the force launch forms the face stresses.

// Rows of C per face axis, and the strain entries the face gradient
// components (x, y, z) enter.
__constant__ int kFaceRows[3][3] = {{0, 5, 4}, {5, 1, 3}, {4, 3, 2}};
__constant__ int kFaceCols[3][3] = {{0, 5, 4}, {5, 1, 3}, {4, 3, 2}};

// P^ax of a cell (its strain e, eigenstrain e0, face gradients g; C its
// stiffness): the strain of its faces along ax with their own gradients
// zero, times the rows of C those faces carry.
__device__ __forceinline__ void p_axis(const double (*C)[6], int ax, const double (&g)[6][3], const double (&e)[6],
                                       const double (&e0)[6], double (&P)[3]) {
    double b[6];
    if (ax == 0) {
        b[0] = -e0[0]; b[1] = e[1] - e0[1]; b[2] = e[2] - e0[2]; b[3] = (e[3] - e0[3]) * 2.;
        b[4] = ((g[4][0] + g[5][0]) / 4. - e0[4]) * 2.; b[5] = ((g[2][0] + g[3][0]) / 4. - e0[5]) * 2.;
    } else if (ax == 1) {
        b[0] = e[0] - e0[0]; b[1] = -e0[1]; b[2] = e[2] - e0[2]; b[3] = ((g[4][1] + g[5][1]) / 4. - e0[3]) * 2.;
        b[4] = (e[4] - e0[4]) * 2.; b[5] = ((g[0][1] + g[1][1]) / 4. - e0[5]) * 2.;
    } else {
        b[0] = e[0] - e0[0]; b[1] = e[1] - e0[1]; b[2] = -e0[2]; b[3] = ((g[2][2] + g[3][2]) / 4. - e0[3]) * 2.;
        b[4] = ((g[0][2] + g[1][2]) / 4. - e0[4]) * 2.; b[5] = (e[5] - e0[5]) * 2.;
    }
    for (int o = 0; o < 3; o++) P[o] = crow(C, kFaceRows[ax][o], b);
}

__device__ __forceinline__ const double (*stiffness(const double* ctab, uint32_t code))[6] {
    return reinterpret_cast<const double (*)[6]>(ctab + ((code & kMatMask) - 1u) * 36u);
}

// The workgroup's LDS copy of every material's constants: the stiffness
// matrices (36 each), then the eigenstrain constants (kEigC each), then
// el_rho, el_mass, el_stiff (kElC each).
constexpr int kGroup = 256;   // threads of a prep or force workgroup
constexpr int kElC = 3;
constexpr int kLdsPerMat = 36 + kEigC + kElC;

__device__ __forceinline__ void load_ctab(double* ctab, const DevMaterial* mats, int nmat) {
    for (int t = threadIdx.x; t < 36 * nmat; t += blockDim.x) ctab[t] = mats[t / 36].cij[(t % 36) / 6][t % 6];
    double* ec = ctab + 36 * nmat;
    for (int t = threadIdx.x; t < kEigC * nmat; t += blockDim.x) {
        const DevMaterial& M = mats[t / kEigC];
        const int q = t % kEigC;
        ec[t] = q == 0 ? M.l100 : q == 1 ? M.l111 : q == 2 ? M.l100a : q == 3 ? M.l111a : q == 4 ? M.l100b
              : q == 5 ? M.l111b : q == 6 ? M.Q11 : q == 7 ? M.Q12 : M.Q44;
    }
    double* lc = ec + kEigC * nmat;
    for (int t = threadIdx.x; t < kElC * nmat; t += blockDim.x) {
        const DevMaterial& M = mats[t / kElC];
        const int q = t % kElC;
        lc[t] = q == 0 ? M.el_rho : q == 1 ? M.el_mass : M.el_stiff;
    }
    __syncthreads();
}

// ---------------------------------------------------------------- prep
// The strain of the u store and the eigenstrain of the stage stores, both
// written out, and the cell's P^x, P^y, P^z; at stage 4 the boundary planes
// of u go to the history.  kGeneral: rotation and the flexoelectric terms
// (the face gradients are written out for the latter).
template <bool kGeneral>
__global__ void __launch_bounds__(256) el_prep_kernel(ElStageArgs a) {
    extern __shared__ double ctab[];   // the materials' constants (load_ctab)
    load_ctab(ctab, a.e.mats, a.f.nmat);
    const int64_t id = static_cast<int64_t>(xcd_group(blockIdx.x, gridDim.x)) * blockDim.x + threadIdx.x;
    if (id >= a.s.nx * a.s.ny * a.s.nz) return;
    int64_t i, j, k;
    cell_ijk(a.s, id, i, j, k);
    double g[6][3], e[6], e0[6] = {0., 0., 0., 0., 0., 0.}, sc[6];
    const uint32_t code = a.s.code[id];
    // the eigenstrain first: its loads then go out with the store's, before
    // any of the launch's writes
    if (a.eig) eigenstrain<kGeneral>(a.e, ctab + 36 * a.f.nmat, id, code, sc, e0);
    cell_grad(a.s, id, i, j, k, g);
    if (kGeneral && a.s.gyz[0]) grad_out(a.s, i, j, k, g);
    strain_of(g, e);
    // the strain array is read by the magnets and ferroelectrics at their own
    // cells (and, for the flexoelectric force, around them: the general form);
    // a download recomputes it everywhere
    if (kGeneral || (code & (kIsFM | kIsAFM | kIsFE))) strain_out(a.s, id, e);
    if (a.eig && a.e0_out) {
        for (int c = 0; c < 6; c++) a.e.e0g[c][id] = e0[c];
        if (a.e.e0c[0] != a.e.e0g[0])
            for (int c = 0; c < 6; c++) a.e.e0c[c][id] = sc[c];
    }
    if (a.h.slot) {
        const int64_t nxy = a.s.nx * a.s.ny, ij = i * a.s.ny + j;
        for (int p = 0; p < kHistPlanes; p++)
            if (k == a.h.planes[p])
                for (int c = 0; c < 3; c++) a.h.slot[(p * 3 + c) * nxy + ij] = a.h.u[c][id];
    }
    double P[3][3] = {{0., 0., 0.}, {0., 0., 0.}, {0., 0., 0.}};
    if (code & kMatMask) {
        const double(*C)[6] = stiffness(ctab, code);
        p_axis(C, 0, g, e, e0, P[0]);
        p_axis(C, 1, g, e, e0, P[1]);
        p_axis(C, 2, g, e, e0, P[2]);
    }
    for (int o = 0; o < 3; o++) {
        a.px[o][id] = P[0][o];
        a.py[o][id] = P[1][o];
        a.pz[o][id] = P[2][o];
    }
}

// ----------------------------------------------------------------- force
// The stress of each face from the P's of its two cells, its gradient (from
// the u store the prep launch read) and the two stiffnesses; dv; the v and
// u RK updates, the next u store into f.us.
// Bound by memory latency: the inputs of a face used to wait for the code
// that says whether it is free.  Here the store, codes and the P's of the y
// and z faces are loaded before any code is known and the z neighbours come
// from the adjacent lanes; the x faces' P's (9 values) are loaded after the
// other axes are done, so that the kernel stays at 126 VGPRs and 4 waves per
// SIMD (with them first: 141 and 3 waves).  1M cells (128x128x64): 95.4 ->
// 86.5 us; 70k cells (45x38x41): 13.9 -> 12.2 us.
// group: the workgroup's index among those of the force.
template <class I>
__device__ __forceinline__ void el_force_group(const ElStageArgs& a, double* ctab, unsigned group) {
    const ElForceArgs& f = a.f;
    load_ctab(ctab, f.mats, f.nmat);
    const I nx = static_cast<I>(f.nx), ny = static_cast<I>(f.ny), nz = static_cast<I>(f.nz);
    const I id = static_cast<I>(group) * kGroup + static_cast<I>(threadIdx.x);
    if (id >= nx * ny * nz) return;
    I i, j, k;
    cell_xyz(a.s.div, id, ny, nz, i, j, k);
    const int stage = f.stage;
    const I ib = i == 0 ? nx - 1 : i - 1, iff = i == nx - 1 ? 0 : i + 1;
    const I jb = j == 0 ? ny - 1 : j - 1, jf = j == ny - 1 ? 0 : j + 1;
    // The reference wraps the forward z neighbour on k == ny - 1
    // (elastic_dynamic_solver.cpp:1247) for the neighbour's stress, not for
    // the face gradient; set-up rejects the grids where that differs from the
    // periodic wrap and reads outside a column.  At k == nz - 1 both wrap
    // (the face is free, or z is periodic and ny == nz), so every index below
    // is inside the arrays.
    const bool odd = k == ny - 1 && k != nz - 1;
    const I kb = k == 0 ? nz - 1 : k - 1, kt = k == nz - 1 ? 0 : k + 1;
    const I col = (i * ny + j) * nz;
    const I nb[6] = {(ib * ny + j) * nz + k, (iff * ny + j) * nz + k, (i * ny + jb) * nz + k,
                     (i * ny + jf) * nz + k, col + kb, odd ? col : col + kt};
    // The codes, store values and P's (but the x faces') of the cell and its
    // neighbours, loaded before any code is known; the z neighbours' from the
    // adjacent lanes as in cell_grad.
    const uint32_t code = ldu(f.code, id);
    double u0[3], un[6][3], Po[3][3], Pn[6][3];
    uint32_t cn[6], ct;
    for (int c = 0; c < 3; c++) u0[c] = ldd(a.s.us[c], id);
    for (int o = 0; o < 3; o++) { Po[1][o] = ldd(a.py[o], id); Po[2][o] = ldd(a.pz[o], id); }
    for (int q = 0; q < 4; q++) {
        cn[q] = ldu(f.code, nb[q]);
        for (int c = 0; c < 3; c++) un[q][c] = ldd(a.s.us[c], nb[q]);
        if (q > 1)
            for (int o = 0; o < 3; o++) Pn[q][o] = ldd(a.py[o], nb[q]);
    }
    const int lane = static_cast<int>(threadIdx.x & 63u);
    const bool gm = lane == 0 || k == 0, gp = lane == 63 || k == nz - 1;
    if (gm) {
        cn[4] = ldu(f.code, nb[4]);
        for (int c = 0; c < 3; c++) un[4][c] = ldd(a.s.us[c], nb[4]);
        for (int o = 0; o < 3; o++) Pn[4][o] = ldd(a.pz[o], nb[4]);
    }
    if (gp) {
        ct = ldu(f.code, col + kt);
        for (int c = 0; c < 3; c++) un[5][c] = ldd(a.s.us[c], col + kt);
    }
    if (gp || odd) {
        cn[5] = ldu(f.code, nb[5]);
        for (int o = 0; o < 3; o++) Pn[5][o] = ldd(a.pz[o], nb[5]);
    }
    for (int c = 0; c < 3; c++) {
        const double ud = lane_up(u0[c]), uu = lane_down(u0[c]);
        const double pd = lane_up(Po[2][c]), pu = lane_down(Po[2][c]);
        if (!gm) { un[4][c] = ud; Pn[4][c] = pd; }
        if (!gp) un[5][c] = uu;
        if (!(gp || odd)) Pn[5][c] = pu;
    }
    const uint32_t cdn = lane_up(code), cup = lane_down(code);
    if (!gm) cn[4] = cdn;
    if (!gp) ct = cup;
    if (!(gp || odd)) cn[5] = cup;
    double dv[3] = {0., 0., 0.};
    if (code & kMatMask) {
        const double(*Cq)[6] = stiffness(ctab, code);
        const bool fr[6] = {(i == 0 && !f.per[0]) || !(cn[0] & kMatMask),
                            (i == nx - 1 && !f.per[0]) || !(cn[1] & kMatMask),
                            (j == 0 && !f.per[1]) || !(cn[2] & kMatMask),
                            (j == ny - 1 && !f.per[1]) || !(cn[3] & kMatMask),
                            (k == 0 && !f.per[2]) || !(cn[4] & kMatMask),
                            (k == nz - 1 && !f.per[2]) || !(ct & kMatMask)};
        const double ih[3] = {f.idx, f.idy, f.idz};
        double d[3][3];
        for (int ax = 2; ax >= 0; ax--) {
            if (ax == 0)
                for (int o = 0; o < 3; o++) {
                    Po[0][o] = ldd(a.px[o], id);
                    Pn[0][o] = ldd(a.px[o], nb[0]);
                    Pn[1][o] = ldd(a.px[o], nb[1]);
                }
            double s1[3] = {0., 0., 0.}, s2[3] = {0., 0., 0.};
            for (int side = 0; side < 2; side++) {
                const int fc = 2 * ax + side;
                double* sf = side ? s2 : s1;
                if (fr[fc]) {
                    // Gaussian traction on a stress-free top face (input_strain_type 3)
                    if (fc == 5 && static_cast<int64_t>(k) == f.trac_k) sf[f.trac_row] = f.trac_amp;
                    continue;
                }
                // the face gradient, across to the face's true neighbour (the
                // value the cell on either side computes for it)
                double fg[3];
                for (int c = 0; c < 3; c++) fg[c] = side ? (un[fc][c] - u0[c]) * ih[ax] : (u0[c] - un[fc][c]) * ih[ax];
                const double(*Cn)[6] = stiffness(ctab, cn[fc]);
                for (int o = 0; o < 3; o++) {
                    const int r = kFaceRows[ax][o];
                    double tq = Po[ax][o], tn = Pn[fc][o];
                    for (int c = 0; c < 3; c++) {
                        const int cc = kFaceCols[ax][c];
                        tq = tq + Cq[r][cc] * fg[c];
                        tn = tn + Cn[r][cc] * fg[c];
                    }
                    sf[o] = (tq + tn) / 2.;
                }
            }
            for (int c = 0; c < 3; c++) d[ax][c] = s2[c] - s1[c];
        }
        const double* lc = ctab + (36 + kEigC) * f.nmat + ((code & kMatMask) - 1) * kElC;
        const double el_rho = lc[0], el_mass = lc[1], el_stiff = lc[2];
        for (int c = 0; c < 3; c++) {
            const double fo = d[0][c] * f.idx + d[1][c] * f.idy + d[2][c] * f.idz;
            // the stored force only matters with stiffness damping
            const double fs = el_stiff != 0. ? ldd(f.fstore[c], id) : 0.;
            if (stage == 2 || stage == 3)
                dv[c] = fo * el_rho + el_mass * ldd(f.v[c], id) + el_stiff * (fo - fs) * 2.;
            else
                dv[c] = fo * el_rho + el_mass * ldd(f.v[c], id) + el_stiff * (fo - fs);
            if (stage == 1) std_(f.fstore[c], id, fo);
        }
    }
    const bool plane = f.liao && k == 0;
    // fourth-order Liao extrapolation of the plane from planes 1..4 of t1..t4
    double bv[3] = {0., 0., 0.};
    if (plane) {
        const I nxy = nx * ny, ij = i * ny + j, pl = 3 * nxy;
        const double w = f.w;
        for (int c = 0; c < 3; c++) {
            const I o = static_cast<I>(c) * nxy + ij;
            bv[c] = (4. * w + 2. * (1. - w)) * ldd(f.hist[0], o) - (6. * w + (1. - w)) * ldd(f.hist[1], pl + o) +
                    (4. * w) * ldd(f.hist[2], 2 * pl + o) - w * ldd(f.hist[3], 3 * pl + o);
        }
    }
    const bool source = static_cast<int64_t>(k) == f.src_k && (code & kMatMask) != 0u;
    for (int c = 0; c < 3; c++) {
        const double du = ldd(f.vs[c], id) * f.dt;
        const double v = ldd(f.v[c], id), u = ldd(f.u[c], id);
        const bool src = source && c == f.src_comp;
        if (stage == 4) {
            const double vn = ldd(f.accv[c], id) + dv[c] * kSixth;
            double un = ldd(f.accu[c], id) + du * kSixth;
            if (plane) un = bv[c];
            if (src) un = f.src_val;
            std_(f.v[c], id, vn);
            std_(f.vs[c], id, vn);
            std_(f.u[c], id, un);
            std_(f.us[c], id, un);
            continue;
        }
        // stages 1-3 set the Liao plane of u itself, the source in its store
        if (plane) std_(f.u[c], id, bv[c]);
        if (stage == 1) {
            std_(f.vs[c], id, v + dv[c] * 0.5);
            std_(f.accv[c], id, v + dv[c] * kSixth);
            std_(f.us[c], id, src ? f.src_val : u + du * 0.5);
            std_(f.accu[c], id, u + du * kSixth);
        } else if (stage == 2) {
            std_(f.vs[c], id, v + dv[c] * 0.5);
            std_(f.accv[c], id, ldd(f.accv[c], id) + dv[c] * kThird);
            std_(f.us[c], id, src ? f.src_val : u + du * 0.5);
            std_(f.accu[c], id, ldd(f.accu[c], id) + du * kThird);
        } else {
            std_(f.vs[c], id, v + dv[c]);
            std_(f.accv[c], id, ldd(f.accv[c], id) + dv[c] * kThird);
            std_(f.us[c], id, src ? f.src_val : u + du);
            std_(f.accu[c], id, ldd(f.accu[c], id) + du * kThird);
        }
    }
}

template <class I>
__global__ void __launch_bounds__(kGroup) el_force_kernel(ElStageArgs a) {
    extern __shared__ double ctab[];   // the materials' constants (load_ctab)
    el_force_group<I>(a, ctab, xcd_group(blockIdx.x, gridDim.x));
}

// The ferromagnet's stage and the elastic force in one launch: the magnet
// reads the strain the prep launch wrote and its own stores, the force reads
// the stress parts of the same launch, and neither reads what the other
// writes.  The magnet's workgroups (over the list of FM cells when some
// cells are not FM) come first: their chain is the longer one.  On 70k cells
// (45x38x41) each launch is mostly latency, and the magnet's 7.8 us hide in
// the force's: 60 steps 7.66 -> 6.34 ms; 128x128x64: 45.5 -> 43.7 ms.
template <bool kMixed>
__global__ void __launch_bounds__(kGroup) el_force_mag_kernel(ElStageArgs a, StageArgs, const uint32_t* ids,
                                                              uint32_t count, unsigned mag_groups) {
    extern __shared__ double ctab[];   // the materials' constants (load_ctab)
    if (blockIdx.x >= mag_groups) {
        el_force_group<uint32_t>(a, ctab, xcd_group(blockIdx.x - mag_groups, gridDim.x - mag_groups));
        return;
    }
    const uint32_t t = blockIdx.x * kGroup + threadIdx.x;
    if (t >= count) return;
    // by value beside the force's, 96 scalar registers spill (128x128x64 with 4
    // layers of magnet 588 us a step, 586 so; 48x48x48 101.9 and 100.3); the force's
    // read like this is slower on small grids (12x10x16: 63 us, 67)
    const StageArgs& m = launch_arg<StageArgs, sizeof(ElStageArgs)>();
    if (ids) fm_point<uint32_t, false, kMixed>(m, ldu(ids, t));
    else fm_point<uint32_t, true, kMixed>(m, t);
}

// -------------------------------------------------------------- boundary
__global__ void __launch_bounds__(256) el_boundary_kernel(ElBoundaryArgs a) {
    const int64_t nxy = a.nx * a.ny, nz = a.nz;
    const int64_t ij = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (ij >= nxy) return;
    const int64_t col = ij * nz;
    auto hist = [&](int plane, int c) { return a.t1[(plane * 3 + c) * nxy + ij]; };
    if (a.mur_bottom) {
        for (int c = 0; c < 3; c++) {
            const double cc = c == 2 ? a.cb_l : a.cb_t;
            if (a.kind < 2) {
                a.us[c][col] = a.u[c][col + 1] + cc * (a.u[c][col] - a.us[c][col + 1]);
            } else {
                const double val = hist(1, c) + cc * (hist(0, c) - a.u[c][col + 1]);
                a.u[c][col] = val;
                a.us[c][col] = val;
            }
        }
    }
    for (int c = 0; c < 3; c++) {
        const double cc = c == 2 ? a.ct_l : a.ct_t;
        const int64_t top = col + nz - 1, below = col + nz - 2;
        if (a.kind < 2) {
            a.us[c][top] = a.u[c][below] + cc * (a.u[c][top] - a.us[c][below]);
        } else {
            const double val = hist(2, c) + cc * (hist(3, c) - a.u[c][below]);
            a.u[c][top] = val;
            a.us[c][top] = val;
        }
    }
    if (a.src_k >= 0 && solid(a.code, col + a.src_k)) {
        const int64_t s = col + a.src_k;
        if (a.kind < 2) {
            a.us[a.src_comp][s] = a.src_val;
        } else {
            a.u[a.src_comp][s] = a.src_val;
            a.us[a.src_comp][s] = a.src_val;
        }
    }
}

unsigned blocks_for(int64_t n) { return static_cast<unsigned>((n + 255) / 256); }

}  // namespace

hipError_t launch_el_strain(const ElStrainArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(el_strain_kernel, dim3(blocks_for(a.nx * a.ny * a.nz)), dim3(256), 0, s, a);
    return hipGetLastError();
}

static size_t el_lds(const ElStageArgs& a) {
    return sizeof(double) * kLdsPerMat * static_cast<size_t>(a.f.nmat > 0 ? a.f.nmat : 1);
}

// Up to 255 materials: 96 KiB of the CU's 160 KiB.
static hipError_t allow_lds(const void* kernel, size_t lds) {
    if (lds <= 65536) return hipSuccess;
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
}

hipError_t launch_el_prep(const ElStageArgs& a, hipStream_t s) {
    const bool general = a.s.rotate || a.e.rotate || a.e.flexo;
    const auto prep = general ? el_prep_kernel<true> : el_prep_kernel<false>;
    const size_t lds = el_lds(a);
    const hipError_t e = allow_lds(reinterpret_cast<const void*>(prep), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(prep, dim3(blocks_for(a.f.nx * a.f.ny * a.f.nz)), dim3(kGroup), lds, s, a);
    return hipGetLastError();
}

hipError_t launch_el_force(const ElStageArgs& a, hipStream_t s) {
    // 32-bit element offsets where they reach
    const bool small = el_narrow(a.f.nx, a.f.ny, a.f.nz, a.f.liao);
    const auto force = small ? el_force_kernel<uint32_t> : el_force_kernel<int64_t>;
    const size_t lds = el_lds(a);
    const hipError_t e = allow_lds(reinterpret_cast<const void*>(force), lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(force, dim3(blocks_for(a.f.nx * a.f.ny * a.f.nz)), dim3(kGroup), lds, s, a);
    return hipGetLastError();
}

// Grids that el_narrow accepts; ids and count as launch_mag_stage.
hipError_t launch_el_force_mag(const ElStageArgs& a, const StageArgs& m, const uint32_t* ids, int64_t count,
                               hipStream_t s) {
    const size_t lds = el_lds(a);
    const auto both = m.mixed ? el_force_mag_kernel<true> : el_force_mag_kernel<false>;
    const hipError_t e = allow_lds(reinterpret_cast<const void*>(both), lds);
    if (e != hipSuccess) return e;
    const unsigned mg = blocks_for(count);
    hipLaunchKernelGGL(both, dim3(mg + blocks_for(a.f.nx * a.f.ny * a.f.nz)), dim3(kGroup), lds, s, a, m, ids,
                       static_cast<uint32_t>(count), mg);
    return hipGetLastError();
}

hipError_t launch_el_boundary(const ElBoundaryArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(el_boundary_kernel, dim3(blocks_for(a.nx * a.ny)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace gf
