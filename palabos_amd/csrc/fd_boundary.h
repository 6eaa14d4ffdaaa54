// Data processors that run after the stream of every step (and once from
// MultiBlock3D::initialize, multiBlock3D.cpp:330-332), on the device:
//
//   * the Neumann-type copies of a boundary's stored value from the cell one
//     step inside it (CopyVelocityFunctional3D, CopyTangentialVelocityFunctional3D,
//     CopyNormalVelocityFunctional3D, CopyDensityFunctional3D;
//     boundaryCondition/neumannCondition3D.hh:116-252), installed for the
//     outflow, neumann, freeslip and normalOutflow boundary types
//     (boundaryInstantiator3D.h:1042-1063, 1097-1102, 1139-1157, 1216-1232);
//   * the finite-difference closures of external velocity edges and corners
//     (OuterVelocityEdgeFunctional3D, OuterVelocityCornerFunctional3D;
//     finiteDifferenceBoundaryProcessor3D.hh:130-329): density from the
//     neighbours inside, the strain rate from one-sided differences of the
//     neighbours' velocities (centred along an edge), and the cell rebuilt as
//     equilibrium plus the off-equilibrium part of that strain rate
//     (IsoThermalBulkDynamics::regularize, isoThermalDynamics.hh:55-69).
//
// Palabos runs the processors one after the other in the order the boundary
// objects were added. The device runs them in four launches (phases): the
// copies of faces and edges, the edge closures, the copies of corners, the
// corner closures. The host checks that no cell is read in the phase that
// writes it and that the phases keep the order of the objects that touch
// (engine.hip, rebuild), so the results are those of the sequential order.
//
// Every neighbour is resolved on the host (ProcNb: a plane, edge or corner cell
// with its stored value, or a plain cell of the block); the neighbour's density and velocity are what its dynamics reports (Cell::computeDensity /
// computeVelocity), from its populations at the current layout parity. A
// plane cell of a wrapped factory is read completed, as its own processor
// leaves it (wrappedLocalBoundaryProcessor3D.hh:41-62).
#pragma once

#include "kernels.h"

namespace plbamd {

enum ProcOp : uint8_t {
    PROC_COPY_VELOCITY = 1,    // CopyVelocityFunctional3D
    PROC_COPY_TANGENTIAL = 2,  // CopyTangentialVelocityFunctional3D: normal components zeroed
    PROC_COPY_NORMAL = 3,      // CopyNormalVelocityFunctional3D: tangential components zeroed
    PROC_COPY_DENSITY = 4,     // CopyDensityFunctional3D
    PROC_EDGE = 5,             // OuterVelocityEdgeFunctional3D
    PROC_CORNER = 6,           // OuterVelocityCornerFunctional3D
};

// A neighbour as the host resolved it: its position, and of a special cell
// (plane, edge, corner) its info and stored value.
struct ProcNb {
    uint32_t cell;      // block-local
    uint32_t value;     // special: index of its stored value
    uint32_t wall;      // link-wall mask
    uint16_t x, y, z;
    uint16_t info;      // special: SpecialCell::info with kNbSpecial; 0: a plain cell
};
constexpr uint16_t kNbSpecial = 0x8000u;

struct ProcCell {
    ProcNb self;        // the processed cell
    ProcNb nb[4];       // copies: nb[0] = cell - n
                        // edges: nb[0] = cell - n1 e1, nb[1] = cell - n2 e2 (e1, e2 the axes after the
                        //        edge's axis), nb[2] / nb[3] = cell +- e along the edge
                        // corners: nb[0..2] = cell - n_x e_x, - n_y e_y, - n_z e_z
    uint8_t op;         // ProcOp
    int8_t n[3];        // outward normal of the boundary (zero along an edge's axis)
};

struct ProcArgs {
    void* arena;
    const BlockGeom* blocks;
    double* values;          // stored boundary values (velocity: 3, density: 1), rewritten by the copies
    const ProcCell* cells;
    uint32_t begin, end;     // the records of this phase
    int parity;              // layout parity of the state the processors act on
    double omega;
};

// What a processor reads of a neighbour, from one load of its populations:
//   rho  Cell::computeDensity: fullRho of the Dirichlet rhoBar for a plane cell
//        (boundaryDynamics.hh:640-679, StoreDensityDynamics :229-233),
//        fullRho(get_rhoBar) otherwise (core/dynamics.hh:278-281, boundaryDynamics.hh:82-87);
//   u    Cell::computeVelocity: the stored velocity of edge, corner and
//        velocity-plane cells (boundaryDynamics.hh:324-330), j / rho of a pressure
//        plane's closure (:776-835), j / rho of the populations otherwise
//        (compute_uLb, momentTemplates3D.h:138-144, with the sequentially summed rhoBar).
template<typename S>
__device__ __forceinline__ void read_nb(const ProcArgs& a, const BlockGeom& g, const ProcNb& c, bool wantRho, bool wantU,
                                        typename Store<S>::T& rho, typename Store<S>::T u[3]) {
    using T = typename Store<S>::T;
    const bool special = (c.info & kNbSpecial) != 0;
    const uint32_t kind = c.info & 3u;
    const bool plane = special && kind == SK_PLANE;
    const bool stored = special && (kind == SK_STORE_VELOCITY || (plane && ((c.info >> 3) & 1u) == PLBAMD_VELOCITY));
    const double* v = a.values + c.value;
    if (wantU && stored) { u[0] = (T)v[0]; u[1] = (T)v[1]; u[2] = (T)v[2]; }
    if (!wantRho && (!wantU || stored)) return;
    T f[19];
    const S* base = reinterpret_cast<const S*>(a.arena) + g.offset;
#pragma unroll
    for (int i = 0; i < 19; ++i)
        f[i] = Store<S>::load(base + pop_index(g, a.parity, c.x, c.y, c.z, i, a.parity ? c.wall : 0u, c.cell));
    if (plane) {
        if ((c.info >> 7) & 1u) complete_plane(f, c.info, v);
        T rhoBar, w[3];
        plane_macroscopic_any(f, c.info, v, rhoBar, w);
        rho = rhoBar + (T)1;
        if (!stored) { u[0] = w[0]; u[1] = w[1]; u[2] = w[2]; }
        return;
    }
    const T rhoBar = rhobar_sum(f);
    rho = rhoBar + (T)1;
    if (!stored) {
        T rb, j[3];
        rhobar_j(f, rb, j);
        const T ir = inv_rho(rhoBar);
        u[0] = j[0] * ir; u[1] = j[1] * ir; u[2] = j[2] * ir;
    }
}

// pi from the velocity gradient g[a][b] = d_a u_b and the density
// (finiteDifferenceBoundaryProcessor3D.hh:162-172, :288-296), order xx xy xz yy yz zz.
template<typename T>
__device__ __forceinline__ void strain_to_pi(const T g[3][3], T rho, T omega, T pi[6]) {
    const T sToPi = -rho / (T)3 / omega;
    pi[0] = (T)2 * g[0][0] * sToPi;
    pi[3] = (T)2 * g[1][1] * sToPi;
    pi[5] = (T)2 * g[2][2] * sToPi;
    pi[1] = (g[0][1] + g[1][0]) * sToPi;
    pi[2] = (g[0][2] + g[2][0]) * sToPi;
    pi[4] = (g[1][2] + g[2][1]) * sToPi;
}

// IsoThermalBulkDynamics::regularize (isoThermalDynamics.hh:55-69) with
// j = rho u and rhoBar = rho - 1, written to the cell's own populations.
template<typename S>
__device__ __forceinline__ void regularize_store(const ProcArgs& a, const BlockGeom& g, const ProcNb& sc,
                                 typename Store<S>::T rho, const typename Store<S>::T u[3],
                                 const typename Store<S>::T pi[6]) {
    using T = typename Store<S>::T;
    T j[3];
    for (int c = 0; c < 3; ++c) j[c] = rho * u[c];
    const T jSqr = j[0] * j[0] + j[1] * j[1] + j[2] * j[2];
    const T rhoBar = rho - (T)1;
    const T ir = inv_rho(rhoBar);
    T f[19];
    f[0] = feq(0, rhoBar, ir, j, jSqr) + pi_to_fneq_generic(0, pi);
#pragma unroll
    for (int i = 1; i <= 9; ++i) {
        f[i] = feq(i, rhoBar, ir, j, jSqr);
        f[i + 9] = feq(i + 9, rhoBar, ir, j, jSqr);
        const T fn = pi_to_fneq_generic(i, pi);
        f[i] += fn;
        f[i + 9] += fn;
    }
    S* base = reinterpret_cast<S*>(a.arena) + g.offset;
#pragma unroll
    for (int i = 0; i < 19; ++i)
        Store<S>::store(base + pop_index(g, a.parity, sc.x, sc.y, sc.z, i, a.parity ? sc.wall : 0u, sc.cell), f[i]);
}

// A wavefront per neighbour: what a record reads (up to four neighbours, each a
// chain of record and population loads and a plane's completion) is under way at
// once, and the lanes of a wavefront complete planes of one orientation. The
// first wavefront then combines and writes. kProcRecords: few lanes per
// wavefront, so that a few hundred records spread over the compute units. (One
// thread per record went through the neighbours one after the other, seven
// chains for an edge cell: 30 us a launch whatever the number of records.)
constexpr int kProcRecords = 16;
template<typename S>
__global__ void __launch_bounds__(256) boundary_processors(ProcArgs a) {
    using T = typename Store<S>::T;
    __shared__ T got[4][4][kProcRecords];
    const int lane = (int)(threadIdx.x & 63u), q = (int)(threadIdx.x >> 6);
    const uint32_t k = a.begin + blockIdx.x * kProcRecords + (uint32_t)lane;
    const bool live = lane < kProcRecords && k < a.end;
    const BlockGeom g = a.blocks[0];     // single-block lattices only (buildProcessors)
    const ProcCell& p = a.cells[live ? k : a.begin];
    const uint8_t op = p.op;
    if (live && q < (op == PROC_EDGE ? 4 : (op == PROC_CORNER ? 3 : 1))) {
        const bool wantRho = op == PROC_COPY_DENSITY || (op == PROC_EDGE && q < 2) || op == PROC_CORNER;
        T r = T(), w[3] = {T(), T(), T()};
        read_nb<S>(a, g, p.nb[q], wantRho, op != PROC_COPY_DENSITY, r, w);
        got[q][0][lane] = r;
#pragma unroll
        for (int c = 0; c < 3; ++c) got[q][1 + c][lane] = w[c];
    }
    __syncthreads();
    if (!live || q != 0) return;
    const ProcNb sc = p.self;
    double* v = a.values + sc.value;
    const T omega = (T)a.omega;
    T rho[4], u[4][3];
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        rho[n] = got[n][0][lane];
#pragma unroll
        for (int c = 0; c < 3; ++c) u[n][c] = got[n][1 + c][lane];
    }
    if (op == PROC_COPY_DENSITY) {
        v[0] = (double)rho[0];
    } else if (op <= PROC_COPY_NORMAL) {
        T w[3] = {u[0][0], u[0][1], u[0][2]};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (op == PROC_COPY_TANGENTIAL && p.n[c] != 0) w[c] = T();
            if (op == PROC_COPY_NORMAL && p.n[c] == 0) w[c] = T();
        }
        v[0] = (double)w[0]; v[1] = (double)w[1]; v[2] = (double)w[2];
    } else {
        const T self[3] = {(T)v[0], (T)v[1], (T)v[2]};
        T gr[3][3], r;
        if (op == PROC_EDGE) {
            const int plane = p.n[0] == 0 ? 0 : (p.n[1] == 0 ? 1 : 2);
            const int d1 = (plane + 1) % 3, d2 = (plane + 2) % 3;
            const T n1 = (T)(-(d1 == 0 ? p.n[0] : d1 == 1 ? p.n[1] : p.n[2]));   // -orientation of the
            const T n2 = (T)(-(d2 == 0 ? p.n[0] : d2 == 1 ? p.n[1] : p.n[2]));   // one-sided differences
            r = (T)0.5 * (rho[1] + rho[0]);
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const T along = (u[2][b] - u[3][b]) / (T)2;      // fd::ctl_diff
                const T g1 = n1 * (-self[b] + u[0][b]);          // -orientation * fd::o1_fwd_diff
                const T g2 = n2 * (-self[b] + u[1][b]);
#pragma unroll
                for (int c = 0; c < 3; ++c) gr[c][b] = c == plane ? along : (c == d1 ? g1 : g2);
            }
        } else {   // PROC_CORNER
            r = (T)1 / (T)3 * (rho[2] + rho[1] + rho[0]);
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int b = 0; b < 3; ++b) gr[c][b] = (T)(-p.n[c]) * (-self[b] + u[c][b]);
        }
        T pi[6];
        strain_to_pi(gr, r, omega, pi);
        regularize_store<S>(a, g, sc, r, self, pi);
    }
}

}  // namespace plbamd
