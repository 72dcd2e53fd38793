// step_kernels.hpp — the unfused step kernels, templated on the arithmetic
// type. One thread per cell, cells linear in x-fastest order so every field
// access of a wavefront is a contiguous, coalesced run.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "physics.hpp"

namespace lbm {

constexpr int kBlock = 256;

struct Pos {
    int x, y, z;
};
__device__ __forceinline__ Pos cell_pos(long c, int nx, int ny) {
    Pos p;
    const long xy = (long)nx * ny;
    p.z = (int)(c / xy);
    const long r = c - (long)p.z * xy;
    p.y = (int)(r / nx);
    p.x = (int)(r - (long)p.y * nx);
    return p;
}
__device__ __forceinline__ long cell_of(int x, int y, int z, int nx, int ny) {
    return ((long)z * ny + y) * nx + x;
}

// Global access as uniform base + 32-bit byte offset, so the compiler can use
// the scalar-base addressing form (one VGPR per address instead of two).
template <typename T>
__device__ __forceinline__ T ldo(const T* base, unsigned boff) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + boff);
}
template <typename T>
__device__ __forceinline__ void sto(T* base, unsigned boff, T v) {
    *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + boff) = v;
}

// A cell by position and index. Off is 32 bits while every array, the 15
// populations together included, stays below 4 GiB: an address is then one
// register next to a scalar base.
template <typename Off>
struct Node {
    int x, y, z;
    Off c;   // (z * ny + y) * nx + x
};
template <typename Off, typename T>
__device__ __forceinline__ T ldn(const T* base, Off o) {
    if constexpr (sizeof(Off) == 4) return ldo(base, o * (unsigned)sizeof(T));
    else return base[o];
}
// NT: non-temporal, for outputs that leave the caches before they are read.
template <bool NT = false, typename Off, typename T>
__device__ __forceinline__ void stn(T* base, Off o, T v) {
    T* p = reinterpret_cast<T*>(reinterpret_cast<char*>(base) + o * (Off)sizeof(T));
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// The node and its six stencil neighbours (xm, xp, ym, yp, zm, zp) under one
// set of tags (kind[face], 0 = periodic): a periodic side wraps, any other
// side clamps to the node itself (nb_index).
template <bool WALLS, typename Off>
__device__ __forceinline__ void stencil(const Node<Off>& p, const int n[3], const int kind[6], Off nb[7]) {
    const Off sx = 1, sy = (Off)(unsigned)n[0], sz = sy * (Off)(unsigned)n[1];
    const Off stride[3] = {sx, sy, sz};
    const int pos[3] = {p.x, p.y, p.z};
    nb[0] = p.c;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const Off span = stride[a] * (Off)(unsigned)(n[a] - 1);
        const bool lo = WALLS && kind[2 * a] != 0, hi = WALLS && kind[2 * a + 1] != 0;
        nb[1 + 2 * a] = pos[a] > 0 ? p.c - stride[a] : p.c + (lo ? (Off)0 : span);
        nb[2 + 2 * a] = pos[a] < n[a] - 1 ? p.c + stride[a] : p.c - (hi ? (Off)0 : span);
    }
}

// Gather the 15 incoming populations of a node from the post-collision buffer
// g: upwind neighbour, or the node's own reflected population at a wall (push
// semantics of src/lbm_solver.tpp:144-192 and HandleBoundaryPoint,
// src/boundary_handler.h:403-426, restated as pull through the host-built slot
// table). rho_prev is the density this node had when those populations were
// produced (moving walls; Fields::wdot holds e_j . u_wall per face and slot).
// WALLS false: every velocity face periodic.
//
// No load waits for another, the slot row's aside: a wavefront without a wall
// cell reads the 15 wrapped upwind neighbours, and one with a wall cell
// selects, per lane and slot, the neighbour or the node's own population.
// (A branch per slot made a wall wavefront a chain of 15 dependent loads.)
template <typename T, bool WALLS, typename Off>
__device__ __forceinline__ void gather(const Fields<T>& f, const BCDesc<T>& bc, const Node<Off>& p, int pull,
                                       T out[kQ]) {
    const T* g = f.g;
    const long vs = f.vs;
    if (!pull) {
#pragma unroll
        for (int j = 0; j < kQ; ++j) out[j] = ldn(g + j * vs, p.c);
        return;
    }
    // Index c + 1 of each axis is the wrapped neighbour at -c.
    const int n[3] = {bc.n[0], bc.n[1], bc.n[2]};
    Off d[3][3];
    {
        Off stride = 1;
        const int pos[3] = {p.x, p.y, p.z};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const Off span = stride * (Off)(unsigned)(n[a] - 1);
            d[a][0] = pos[a] < n[a] - 1 ? stride : (Off)0 - span;
            d[a][1] = 0;
            d[a][2] = pos[a] > 0 ? (Off)0 - stride : span;
            stride *= (Off)(unsigned)n[a];
        }
    }
    const int cls = WALLS ? node_class(p.x, p.y, p.z, n[0], n[1], n[2]) : 0;
    if (!WALLS || __builtin_amdgcn_ballot_w64(cls != 0) == 0) {
#pragma unroll
        for (int j = 0; j < kQ; ++j)
            out[j] = ldn(g + j * vs, (Off)(p.c + d[0][cx(j) + 1] + d[1][cy(j) + 1] + d[2][cz(j) + 1]));
        return;
    }
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4* rp = reinterpret_cast<const u32x4*>(f.slots + cls * kSlotRow);
    const u32x4 r0 = rp[0], r1 = rp[1];
    const uint32_t words[8] = {r0[0], r0[1], r0[2], r0[3], r1[0], r1[1], r1[2], r1[3]};
    uint16_t e[kQ];
#pragma unroll
    for (int j = 0; j < kQ; ++j) {
        e[j] = (uint16_t)(words[j >> 1] >> (16 * (j & 1)));
        const Off nb = p.c + d[0][cx(j) + 1] + d[1][cy(j) + 1] + d[2][cz(j) + 1];
        const bool stream = slot_kind(e[j]) == SLOT_STREAM;
        out[j] = ldn(g, (Off)(stream ? (Off)j * (Off)vs + nb : (Off)slot_src(e[j]) * (Off)vs + p.c));
    }
    if (f.wdot) {
        const T rho_prev = bc.rho_base + ldn(f.rho, p.c);
        T dot[kQ];
#pragma unroll
        for (int j = 0; j < kQ; ++j) dot[j] = f.wdot[slot_face(e[j]) * kSlotRow + j];
#pragma unroll
        for (int j = 0; j < kQ; ++j) {
            const T moved = out[j] + T(6.0) * rho_prev * T(wgt(j)) * dot[j];
            out[j] = slot_kind(e[j]) == SLOT_BOUNCE ? moved : out[j];
        }
    }
}

// Ghosts of a node's stencil values, v[i] as `stencil` numbers them: the values
// beyond a wall replace what the stencil read there. Called under a branch
// that only wavefronts with a cell on a wall take, after every load is issued:
// with the selects in line, the wall constants and lane masks of all components
// spilled 90 scalar registers and the FP64 Q kernel held 202 vector registers.
template <typename T>
__device__ __forceinline__ void q_ghosts(const BCDesc<T>& bc, const int pos[3], int c, T v[7]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) q_pair(bc, a, c, pos[a], v[1 + 2 * a], v[0], v[2 + 2 * a], v[1 + 2 * a], v[2 + 2 * a]);
}
template <typename T>
__device__ __forceinline__ void u_ghosts(const BCDesc<T>& bc, const int pos[3], int comp, T v[7]) {
#pragma unroll
    for (int a = 0; a < 3; ++a) u_pair(bc, a, comp, pos[a], v[1 + 2 * a], v[0], v[2 + 2 * a], v[1 + 2 * a], v[2 + 2 * a]);
}
// Whether a cell lies on the first or last plane of an axis with a wall.
__device__ __forceinline__ bool on_wall(const int pos[3], const int n[3], const int qkind[6], const int ukind[6]) {
    bool on = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const bool walls = (qkind[2 * a] | qkind[2 * a + 1] | ukind[2 * a] | ukind[2 * a + 1]) != 0;
        on |= walls & ((pos[a] == 0) | (pos[a] == n[a] - 1));
    }
    return on;
}

// ---- Q update ----------------------------------------------------------------
// QTensorSolver::StepAndSetupBodyForce (src/qtensor_solver.tpp:50-147).
// One cell. `own` false stores the stresses only (a halo cell of a region
// pass whose Q^{n+1} and Ericksen force belong to another launch).
//
// The stresses handed to the force kernel are Sigma and Tau in FP64. FP32
// stores the eight independent components of the divergence form instead
// (stress_sets; zz = -xx - yy), in the same arrays: the force then needs 20
// neighbour values rather than 52 and no Q^{n+1} (force kernel at 97x75x113:
// 31.1 -> 26.3 us, at 256^3: 727 -> 557 us; FP64 keeps the reference's bits).
//
// Every load is issued before the first use, and the ghosts are patched after
// the loads under a branch that only wavefronts with a cell on a wall take
// (q_ghosts): with a branch per component and axis the loads of each component
// waited for the arithmetic of the one before, eight memory latencies in a
// row. Bound by latency on small grids and by the caches on large ones. With
// force_lbm_cell and the block orders of CellGrid, a step of the two kernels
// went from 23.7 to 9.9 us at 32^3 FP64, 48.6 to 29.7 us (FP64) and 30.6 to 14.7
// us (FP32) on a 20x100x100 channel, 400 to 287 us on a 150x130x100 FP64 channel
// and 2.82 to 2.41 ms at 256^3 FP64.
template <typename T>
__device__ __forceinline__ void settle(T& x) {
    if constexpr (sizeof(T) == 8) asm volatile("" : "+v"(x));
}
template <bool WALLS, bool NT, typename T, typename Off>
__device__ __forceinline__ void qstep_cell(const Fields<T>& f, const BCDesc<T>& bc, const Phys<T>& k,
                                           const Node<Off>& p, bool own) {
    const int pos[3] = {p.x, p.y, p.z};
    // Q stencil neighbours (Q tags), velocity neighbours (velocity tags).
    Off qs[7], us[7];
    stencil<WALLS>(p, bc.n, bc.qkind, qs);
    stencil<WALLS>(p, bc.n, bc.ukind, us);
    T Q[5], u[3], g[3][3], w[3][7], v[5][7];
#pragma unroll
    for (int A = 0; A < 3; ++A)
#pragma unroll
        for (int i = 0; i < 7; ++i) w[A][i] = ldn(f.u[A], us[i]);
#pragma unroll
    for (int m = 0; m < 5; ++m)
#pragma unroll
        for (int i = 0; i < 7; ++i) v[m][i] = ldn(f.q[m], qs[i]);
#pragma unroll
    for (int m = 0; m < 5; ++m) Q[m] = v[m][0];
    const bool wall_wave = WALLS && __builtin_amdgcn_ballot_w64(on_wall(pos, bc.n, bc.qkind, bc.ukind)) != 0;
    if (wall_wave) {
#pragma unroll
        for (int A = 0; A < 3; ++A) u_ghosts(bc, pos, A, w[A]);
    }
#pragma unroll
    for (int A = 0; A < 3; ++A) {
        u[A] = w[A][0];
#pragma unroll
        for (int B = 0; B < 3; ++B) g[A][B] = (w[A][2 + 2 * B] - w[A][1 + 2 * B]) / T(2.0);
    }
    QRates<T> r;
    q_rates(k, Q, g, r);
#pragma unroll
    for (int i = 0; i < 5; ++i) settle(r.E[i]);
#pragma unroll
    for (int i = 0; i < 3; ++i) settle(r.W[i]);
#pragma unroll
    for (int m = 0; m < 5; ++m) {
        if (wall_wave && bc.q_ghosts) q_ghosts(bc, pos, m, v[m]);   // otherwise the clamped value is the ghost
        q_component(k, m, Q[m], u, q_deriv<T, true>(bc, m, pos, Q[m], v[m][1], v[m][2], v[m][3], v[m][4], v[m][5], v[m][6]), r);
        settle(r.H[m]);
        settle(r.advc[m]);
    }
    T ta[3], fe[3];
    if constexpr (sizeof(T) == 4) {
        T rate[5], pxy[6], pz[2];
        q_finish(k, Q, r, ta, fe, [&](int c, T rc, T) { rate[c] = rc; });
        stress_sets(k, Q, r.H, rate, pxy, pz);
#pragma unroll
        for (int m = 0; m < 5; ++m) stn<NT>(f.sig[m], p.c, pxy[m]);
        stn<NT>(f.tau[0], p.c, pxy[5]);
        stn<NT>(f.tau[1], p.c, pz[0]);
        stn<NT>(f.tau[2], p.c, pz[1]);
        if (own) {
#pragma unroll
            for (int m = 0; m < 5; ++m) stn<NT>(f.qn[m], p.c, Q[m] + k.dt * rate[m]);
        }
    } else {
        q_finish(k, Q, r, ta, fe, [&](int c, T rate, T sc) {
            stn<NT>(f.sig[c], p.c, sc);
            if (own) stn<NT>(f.qn[c], p.c, Q[c] + k.dt * rate);
        });
#pragma unroll
        for (int m = 0; m < 3; ++m) stn<NT>(f.tau[m], p.c, ta[m]);
    }
    if (own) {
#pragma unroll
        for (int m = 0; m < 3; ++m) stn<NT>(f.F[m], p.c, fe[m]);
    }
}

// One thread per cell, cells linear; positions by multiplication (the
// compiler's 64-bit division is some 150 instructions, three times a cell).
//
// Block order: the hardware deals blocks to the 8 XCDs in turn. In plain order
// (run 0) neighbouring planes are read by every XCD; in runs of consecutive
// cells per XCD, each plane is fetched into one L2. Runs pay while the arrays
// of a step live in the caches: at arrays of 3.3 to 8.4 MB they took FP32
// steps from 70.8 to 51.3 us (97x75x113) and 140 to 131 us (128^3), FP64 from
// 80 to 66 us (96x80x64). From 12 MB on the 8 distant streams cost more HBM
// than they save: 128^3 FP64 310 -> 324 us, 256^3 FP64 2.56 -> 2.92 ms. With
// runs, blocks of 128 threads spread small grids over more CUs (32^3 FP64 12.0
// -> 10.6 us) and are within 1% elsewhere; in plain order they lose up to 12%.
struct CellGrid {
    FastDiv by_plane, by_nx;
    unsigned plane, nx, cells;
    unsigned run;   // blocks per XCD, 0: plain order
    unsigned threads, blocks;
};
constexpr size_t kRunBytes = 9u << 20;   // arrays up to this size take runs
template <typename T>
CellGrid cell_grid(const int n[3]) {
    CellGrid g{};
    g.plane = (unsigned)n[0] * (unsigned)n[1];
    g.nx = (unsigned)n[0];
    g.cells = g.plane * (unsigned)n[2];
    g.by_plane = fast_div(g.plane);
    g.by_nx = fast_div(g.nx);
    const bool runs = (size_t)g.cells * sizeof(T) <= kRunBytes;
    g.threads = runs ? kBlock / 2 : kBlock;
    g.blocks = (g.cells + g.threads - 1) / g.threads;
    if (runs) {
        g.run = (g.blocks + 7) / 8;
        g.blocks = g.run * 8;
    }
    return g;
}
// This thread's cell; cg.cells or more: none.
__device__ __forceinline__ unsigned thread_cell(const CellGrid& g) {
    const unsigned b = g.run ? (blockIdx.x & 7) * g.run + (blockIdx.x >> 3) : blockIdx.x;
    return b * g.threads + threadIdx.x;
}
template <typename Off>
__device__ __forceinline__ Node<Off> node_at(const CellGrid& g, unsigned c) {
    const unsigned z = g.by_plane.div(c), r = c - z * g.plane, y = g.by_nx.div(r);
    return {(int)(r - y * g.nx), (int)y, (int)z, (Off)c};
}

// The FP32 form with walls on small arrays is held to five wavefronts per SIMD:
// left alone, the 64-bit sums of stress_sets (and the wall constants) take it from
// 79 to 117 registers, and 20x100x100 from 14.7 to 14.9 us a step, 64^3 from 15.7
// to 16.0. The other forms are even or slower so (128^3 periodic 121.9 -> 122.4).
template <typename T, bool WALLS, bool NT, int ADV, typename Off>
__global__ void __launch_bounds__(kBlock, sizeof(T) == 4 && WALLS && !NT ? 5 : 0)
qstep_kernel(Fields<T> f, BCDesc<T> bc, Phys<T> k, CellGrid cg) {
    k.advection = ADV;
    const unsigned c = thread_cell(cg);
    if (c >= cg.cells) return;
    qstep_cell<WALLS, NT>(f, bc, k, node_at<Off>(cg, c), true);
}

// ---- body force and collide-stream ----------------------------------------
// Both forms add the active and passive force to the Ericksen force in F.
// FP64: differences of Q^{n+1}, Sigma and Tau in the reference's order. The
// stencil's clamped value is the ghost of Q too, unless GHOSTS (see
// BCDesc::q_ghosts). The velocity is read where friction uses it.
template <bool WALLS, bool GHOSTS, typename T, typename Off>
__device__ __forceinline__ void force_differences(const Fields<T>& f, const BCDesc<T>& bc, const Phys<T>& k,
                                                  const Node<Off>& p, T F[3]) {
    T u[3] = {T(0), T(0), T(0)};
    if (k.mu != T(0)) {
#pragma unroll
        for (int m = 0; m < 3; ++m) u[m] = ldn(f.u[m], p.c);
    }
    const int pos[3] = {p.x, p.y, p.z};
    Off nb[7];
    stencil<WALLS>(p, bc.n, bc.qkind, nb);
    T v[13][7];
#pragma unroll
    for (int m = 0; m < 13; ++m) {
        const T* a = m < 5 ? f.q[m] : (m < 10 ? f.sig[m - 5] : f.tau[m - 10]);
#pragma unroll
        for (int i = 0; i < 7; ++i) v[m][i] = ldn(a, nb[i]);
    }
    T dQ[5][3], dS[8][3];
#pragma unroll
    for (int m = 0; m < 5; ++m) {
        const Deriv<T> d =
            q_deriv<T, !GHOSTS>(bc, m, pos, v[m][0], v[m][1], v[m][2], v[m][3], v[m][4], v[m][5], v[m][6]);
#pragma unroll
        for (int a = 0; a < 3; ++a) dQ[m][a] = d.d[a];
    }
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
        for (int a = 0; a < 3; ++a) dS[m][a] = (v[5 + m][2 + 2 * a] - v[5 + m][1 + 2 * a]) / T(2.0);
    const T fe[3] = {F[0], F[1], F[2]};
    body_force(k, dQ, dS, u, fe, F);
}

// FP32: the divergence form, from the components qstep_cell stored.
template <bool WALLS, bool GHOSTS, typename T, typename Off>
__device__ __forceinline__ void force_divergence(const Fields<T>& f, const BCDesc<T>& bc, const Phys<T>& k,
                                                 const Node<Off>& p, T F[3]) {
    Off nb[7];
    stencil<WALLS>(p, bc.n, bc.qkind, nb);
    // Array of component b of axis a's set: x (xx, yx, zx), y (xy, yy, zy), z (xz, yz, then zz = -xx - yy).
    const T* const sets[3][4] = {{f.sig[0], f.sig[1], f.sig[2], nullptr},
                                 {f.sig[3], f.sig[4], f.tau[0], nullptr},
                                 {f.tau[1], f.tau[2], f.sig[0], f.sig[4]}};
    T v[3][4][2];
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < (a < 2 ? 3 : 4); ++b)
#pragma unroll
            for (int side = 0; side < 2; ++side) v[a][b][side] = ldn(sets[a][b], nb[1 + 2 * a + side]);
    T d[3][3];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        d[0][b] = v[0][b][1] - v[0][b][0];
        d[1][b] = v[1][b][1] - v[1][b][0];
    }
    d[2][0] = v[2][0][1] - v[2][0][0];
    d[2][1] = v[2][1][1] - v[2][1][0];
    d[2][2] = (v[2][2][0] - v[2][2][1]) + (v[2][3][0] - v[2][3][1]);
    if constexpr (GHOSTS) {
        // Where the ghost of Q is not the value beyond the face that the
        // stresses use (anchoring; a periodic high face opposite a wall), the
        // set there holds -alpha times the wrong Q. The sets' Q components:
        constexpr int qc[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, -1}};
        const int pos[3] = {p.x, p.y, p.z};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (bc.qkind[2 * a] == QB_PERIODIC) continue;
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                if (pos[a] != (side ? bc.n[a] - 1 : 0)) continue;
                const int face = 2 * a + side;
                const T sign = side ? -k.alpha : k.alpha;   // -alpha, and minus at the low side
                auto off_by = [&](int c) {
                    const T q0 = ldn(f.q[c], p.c);
                    return (bc.qkind[face] == QB_ANCHOR ? T(2.0) * bc.anchor[face][c] - q0 : q0) - ldn(f.q[c], nb[1 + face]);
                };
#pragma unroll
                for (int b = 0; b < 3; ++b)
                    d[a][b] += sign * (qc[a][b] >= 0 ? off_by(qc[a][b]) : -(off_by(0) + off_by(3)));
            }
        }
    }
    T u[3] = {T(0), T(0), T(0)};
    if (k.mu != T(0)) {
#pragma unroll
        for (int b = 0; b < 3; ++b) u[b] = ldn(f.u[b], p.c);
    }
#pragma unroll
    for (int b = 0; b < 3; ++b) F[b] += T(0.5) * ((d[0][b] + d[1][b]) + d[2][b]) - k.mu * u[b];
}

// SetActiveStressAndComputeBodyForce (src/qtensor_solver.tpp:154-217) and
// LatticeBoltzmannStep (src/lbm_solver.tpp:89-224) at one node. Fusing the two
// is the merge the reference documents as valid (src/qtensor_solver.tpp:219-247):
// the force at a node feeds only that node's collision.
// One cell. UN: the velocity goes to un (fused-step buffers, where u still
// holds u^{n-1} for other cells) instead of replacing u in place. Loads first,
// as in qstep_cell.
template <typename T, bool SHIFTED, bool UN, bool WALLS, bool GHOSTS, bool NT, typename Off>
__device__ __forceinline__ void force_lbm_cell(const Fields<T>& f, const BCDesc<T>& bc, const Phys<T>& k,
                                               const Node<Off>& p, int flags, int pull) {
    T pop[kQ], F[3];
    if (flags & FL_LBM) gather<T, WALLS>(f, bc, p, pull, pop);
#pragma unroll
    for (int m = 0; m < 3; ++m) F[m] = ldn(f.F[m], p.c);   // the Ericksen force, or the whole force
    if (flags & FL_FORCE) {
        if (k.force_full) {
            if constexpr (sizeof(T) == 4) force_divergence<WALLS, GHOSTS>(f, bc, k, p, F);
            else force_differences<WALLS, GHOSTS>(f, bc, k, p, F);
        }
        if (flags & FL_STORE_F) {
#pragma unroll
            for (int m = 0; m < 3; ++m) stn(f.F[m], p.c, F[m]);
        }
    }
    if (!(flags & FL_LBM)) return;

    T rho_st, u[3];   // the density in its stored form (rho - BCDesc::rho_base)
    if constexpr (SHIFTED) collide_shifted(k, pop, F, rho_st, u);
    else collide_plain(k, pop, F, rho_st, u);
    if (flags & FL_STORE_RHO) stn(f.rho, p.c, rho_st);
    T* const* uo = UN ? f.un : f.u;
#pragma unroll
    for (int m = 0; m < 3; ++m) stn<NT>(uo[m], p.c, u[m]);
#pragma unroll
    for (int j = 0; j < kQ; ++j) stn<NT>(f.gn + j * f.vs, p.c, pop[j]);
}

// FLAGS is a template argument so that the step's own combination is one
// straight run from the loads to the stores.
template <typename T, bool SHIFTED, bool WALLS, bool GHOSTS, bool NT, int FLAGS, typename Off>
__global__ void __launch_bounds__(kBlock)
force_lbm_kernel(Fields<T> f, BCDesc<T> bc, Phys<T> k, CellGrid cg, int store, int pull) {
    const unsigned c = thread_cell(cg);
    if (c >= cg.cells) return;
    force_lbm_cell<T, SHIFTED, false, WALLS, GHOSTS, NT>(f, bc, k, node_at<Off>(cg, c),
                                               FLAGS | (store & (FL_STORE_F | FL_STORE_RHO)), pull);
}

template <typename T, bool WALLS, typename Off>
__global__ void __launch_bounds__(kBlock)
stream_only_kernel(Fields<T> f, BCDesc<T> bc, CellGrid cg, int pull, T* out) {
    const unsigned c = thread_cell(cg);
    if (c >= cg.cells) return;
    const Node<Off> p = node_at<Off>(cg, c);
    T pop[kQ];
    gather<T, WALLS>(f, bc, p, pull, pop);
#pragma unroll
    for (int j = 0; j < kQ; ++j) stn(out + j * f.vs, p.c, pop[j]);
}

// ---- FP64 diagnostics ---------------------------------------------------------
// SimIO::Log sums (src/sim_io.cc:78-109) and TotalNematicFreeEnergy
// (src/analysis_fields.h:39-72, Laplacian with the Neumann clamp, neighbour
// order xp, xm, yp, ym, zp, zm; density from src/analysis_fields.cc:38-57).
constexpr int kDiag = 10;
template <typename T>
__global__ void __launch_bounds__(kBlock)
diag_partial_kernel(Fields<T> f, BCDesc<T> bc, Phys<double> k, long V, double* uprev, double* partials) {
    __shared__ double red[kBlock / 64][kDiag];
    double acc[kDiag] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int nx = bc.n[0], ny = bc.n[1], nz = bc.n[2];
    for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < V; c += (long)gridDim.x * blockDim.x) {
        const double r = (sizeof(T) == 4 ? k.rho0 : 0.0) + (double)f.rho[c];
        const double ux = (double)f.u[0][c], uy = (double)f.u[1][c], uz = (double)f.u[2][c];
        acc[0] += r;
        acc[1] += r * ux;
        acc[2] += r * uy;
        acc[3] += r * uz;
        const double u2 = ux * ux + uy * uy + uz * uz;
        acc[4] += 0.5 * r * u2;
        const double dx = ux - uprev[c], dy = uy - uprev[V + c], dz = uz - uprev[2 * V + c];
        acc[5] += dx * dx + dy * dy + dz * dz;
        acc[6] += u2;
        acc[7] = u2 > acc[7] ? u2 : acc[7];
        uprev[c] = ux;
        uprev[V + c] = uy;
        uprev[2 * V + c] = uz;
        if (!isfinite(r) || !isfinite(ux) || !isfinite(uy) || !isfinite(uz)) acc[9] += 1.0;

        const Pos p = cell_pos(c, nx, ny);
        const int xm = nb_index(p.x, -1, nx, bc.qkind[0] == QB_PERIODIC, bc.qkind[1] == QB_PERIODIC);
        const int xp = nb_index(p.x, +1, nx, bc.qkind[0] == QB_PERIODIC, bc.qkind[1] == QB_PERIODIC);
        const int ym = nb_index(p.y, -1, ny, bc.qkind[2] == QB_PERIODIC, bc.qkind[3] == QB_PERIODIC);
        const int yp = nb_index(p.y, +1, ny, bc.qkind[2] == QB_PERIODIC, bc.qkind[3] == QB_PERIODIC);
        const int zm = nb_index(p.z, -1, nz, bc.qkind[4] == QB_PERIODIC, bc.qkind[5] == QB_PERIODIC);
        const int zp = nb_index(p.z, +1, nz, bc.qkind[4] == QB_PERIODIC, bc.qkind[5] == QB_PERIODIC);
        double Q[5], lap[5];
#pragma unroll
        for (int m = 0; m < 5; ++m) {
            const T* v = f.q[m];
            Q[m] = (double)v[c];
            lap[m] = (double)v[cell_of(xp, p.y, p.z, nx, ny)] + (double)v[cell_of(xm, p.y, p.z, nx, ny)]
                   + (double)v[cell_of(p.x, yp, p.z, nx, ny)] + (double)v[cell_of(p.x, ym, p.z, nx, ny)]
                   + (double)v[cell_of(p.x, p.y, zp, nx, ny)] + (double)v[cell_of(p.x, p.y, zm, nx, ny)]
                   - 6.0 * Q[m];
        }
        const double Qxx = Q[0], Qxy = Q[1], Qxz = Q[2], Qyy = Q[3], Qyz = Q[4];
        const double TrQ2 = 2.0 * (Qxx * Qxx + Qxx * Qyy + Qyy * Qyy + Qxy * Qxy + Qxz * Qxz + Qyz * Qyz);
        const double third = 1.0 / 3.0;
        const double Q2xx = Qxx * Qxx + Qxy * Qxy + Qxz * Qxz - third * TrQ2;
        const double Q2xy = Qxx * Qxy + Qxy * Qyy + Qxz * Qyz;
        const double Q2xz = Qxy * Qyz - Qxz * Qyy;
        const double Q2yy = Qxy * Qxy + Qyy * Qyy + Qyz * Qyz - third * TrQ2;
        const double Q2yz = Qxy * Qxz - Qyz * Qxx;
        const double TrQ3 = 2.0 * Qxx * Q2xx + 2.0 * Qyy * Q2yy + Qxx * Q2yy + Qyy * Q2xx
                          + 2.0 * (Qxy * Q2xy + Qxz * Q2xz + Qyz * Q2yz);
        const double QlapQ = 2.0 * Qxx * lap[0] + 2.0 * Qyy * lap[3] + Qxx * lap[3] + Qyy * lap[0]
                           + 2.0 * (Qxy * lap[1] + Qxz * lap[2] + Qyz * lap[4]);
        acc[8] += 0.5 * k.A * TrQ2 + (k.B / 3.0) * TrQ3 + 0.25 * k.C * TrQ2 * TrQ2 - 0.5 * k.L * QlapQ;
    }
    // Wavefront reduction (64 lanes), then across the block's wavefronts.
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int m = 0; m < kDiag; ++m) {
        double v = acc[m];
        for (int off = 32; off > 0; off >>= 1) {
            const double o = __shfl_down(v, off, 64);
            v = (m == 7) ? (o > v ? o : v) : v + o;
        }
        if (lane == 0) red[wave][m] = v;
    }
    __syncthreads();
    if (threadIdx.x < kDiag) {
        const int m = threadIdx.x;
        double v = red[0][m];
        for (int w = 1; w < kBlock / 64; ++w) v = (m == 7) ? (red[w][m] > v ? red[w][m] : v) : v + red[w][m];
        partials[(long)blockIdx.x * kDiag + m] = v;
    }
}

// The blocks' partial sums, one wavefront per quantity. (One thread per
// quantity walked up to 1024 of them in a chain, which was most of the
// diagnostics' time: 261 -> 85 us per call at 128^3 in FP64, 219 -> 46 us at
// 60 x 100 x 60.)
template <int Unused = 0>
__global__ void __launch_bounds__(64 * kDiag) diag_final_kernel(const double* partials, int nblocks, double* out) {
    const int lane = threadIdx.x & 63, m = threadIdx.x >> 6;
    double v = 0.0;
    for (int b = lane; b < nblocks; b += 64) {
        const double x = partials[(long)b * kDiag + m];
        v = (m == 7) ? (x > v ? x : v) : v + x;
    }
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_down(v, off, 64);
        v = (m == 7) ? (o > v ? o : v) : v + o;
    }
    if (lane == 0) out[m] = v;
}

// QtensorToOrderDirector (src/analysis_fields.cc:59-93) in FP64.
template <typename T>
__global__ void __launch_bounds__(kBlock)
order_director_kernel(Fields<T> f, long c0, long n, double* order, double* director) {
    // The directors leave through LDS, so that a wavefront writes whole lines
    // (the target may be host memory).
    __shared__ double out[3 * kBlock];
    const long first = (long)blockIdx.x * kBlock;
    const int t = threadIdx.x, cells = (int)min((long)kBlock, n - first);
    const long c = c0 + first + min(t, cells - 1);
    const double Qxx = f.q[0][c], Qxy = f.q[1][c], Qxz = f.q[2][c], Qyy = f.q[3][c], Qyz = f.q[4][c];
    const double pp = Qxx * Qxx + Qxx * Qyy + Qyy * Qyy + Qxy * Qxy + Qxz * Qxz + Qyz * Qyz;
    const double qd = -(Qxx + Qyy) * (Qxx * Qyy - Qxy * Qxy) - Qyy * Qxz * Qxz - Qxx * Qyz * Qyz + 2 * Qxy * Qxz * Qyz;
    const double r = 2.0 * sqrt(pp / 3.0);
    double arg = 4 * qd / (r * r * r);
    arg = arg < -1.0 ? -1.0 : (arg > 1.0 ? 1.0 : arg);
    const double S = r * cos(1.0 / 3.0 * acos(arg));
    double nxv = Qxz * (Qyy - S) - Qxy * Qyz;
    double nyv = Qyz * (Qxx - S) - Qxy * Qxz;
    double nzv = Qxy * Qxy - (Qxx - S) * (Qyy - S);
    const double inv = 1.0 / sqrt(nxv * nxv + nyv * nyv + nzv * nzv);
    if (t < cells) order[first + t] = S;
    out[3 * t + 0] = nxv * inv;
    out[3 * t + 1] = nyv * inv;
    out[3 * t + 2] = nzv * inv;
    __syncthreads();
    for (int i = t; i < 3 * cells; i += kBlock) director[3 * first + i] = out[i];
}

// ---- launchers ---------------------------------------------------------------
inline unsigned grid_for(long V) { return (unsigned)((V + kBlock - 1) / kBlock); }

// fn(walls, offset) with the kernels' template arguments: whether any face has
// a wall, and the index type (Node).
template <typename T, typename F>
void with_step_form(const BCDesc<T>& bc, long vs, F&& fn) {
    const bool narrow = (size_t)kQ * vs * sizeof(T) < (1ull << 32);
    bool walls = false;
    for (int face = 0; face < 6; ++face)
        walls = walls || bc.qkind[face] != QB_PERIODIC || bc.ukind[face] != UB_PERIODIC;
    auto with_offset = [&](auto w) {
        if (narrow) fn(w, 0u);
        else fn(w, (size_t)0);
    };
    if (walls) with_offset(std::true_type{});
    else with_offset(std::false_type{});
}

template <typename T>
void launch_qstep(const Fields<T>& f, const BCDesc<T>& bc, const Phys<T>& k, hipStream_t s) {
    const CellGrid cg = cell_grid<T>(bc.n);
    with_step_form(bc, f.vs, [&](auto w, auto off) {
        auto go = [&](auto nt, auto adv) {
            hipLaunchKernelGGL((qstep_kernel<T, decltype(w)::value, decltype(nt)::value, decltype(adv)::value, decltype(off)>),
                               dim3(cg.blocks), dim3(cg.threads), 0, s, f, bc, k, cg);
        };
        auto with_adv = [&](auto nt) {
            if (k.advection) go(nt, std::integral_constant<int, 1>{});
            else go(nt, std::integral_constant<int, 0>{});
        };
        if (cg.run) with_adv(std::false_type{});
        else with_adv(std::true_type{});
    });
}

template <typename T, bool SHIFTED>
void launch_force_lbm(const Fields<T>& f, const BCDesc<T>& bc, const Phys<T>& k, int flags, int pull,
                      hipStream_t s) {
    const CellGrid cg = cell_grid<T>(bc.n);
    const int store = flags & (FL_STORE_F | FL_STORE_RHO);
    with_step_form(bc, f.vs, [&](auto w, auto off) {
        constexpr bool walls = decltype(w)::value;
        auto launch = [&](auto parts, auto ghosts, auto nt) {
            hipLaunchKernelGGL((force_lbm_kernel<T, SHIFTED, walls, decltype(ghosts)::value, decltype(nt)::value,
                                                 decltype(parts)::value, decltype(off)>),
                               dim3(cg.blocks), dim3(cg.threads), 0, s, f, bc, k, cg, store, pull);
        };
        auto go = [&](auto parts, auto nt) {
            if constexpr (walls && (decltype(parts)::value & FL_FORCE) != 0) {
                if (bc.q_ghosts) return launch(parts, std::true_type{}, nt);
            }
            launch(parts, std::false_type{}, nt);
        };
        constexpr std::integral_constant<int, FL_FORCE | FL_LBM> both{};
        switch (flags & (FL_FORCE | FL_LBM)) {
            case FL_FORCE: go(std::integral_constant<int, FL_FORCE>{}, std::false_type{}); break;
            case FL_LBM: go(std::integral_constant<int, FL_LBM>{}, std::false_type{}); break;
            default:
                if (cg.run) go(both, std::false_type{});
                else go(both, std::true_type{});
                break;
        }
    });
}

template <typename T>
void launch_stream_only(const Fields<T>& f, const BCDesc<T>& bc, int pull, T* out, hipStream_t s) {
    const CellGrid cg = cell_grid<T>(bc.n);
    with_step_form(bc, f.vs, [&](auto w, auto off) {
        hipLaunchKernelGGL((stream_only_kernel<T, decltype(w)::value, decltype(off)>), dim3(cg.blocks),
                           dim3(cg.threads), 0, s, f, bc, cg, pull, out);
    });
}

template <typename T>
void launch_diagnostics(const Fields<T>& f, const BCDesc<T>& bc, const Phys<double>& k, long V, double* uprev,
                        double* partials, int nblocks, double* out, hipStream_t s) {
    hipLaunchKernelGGL(diag_partial_kernel<T>, dim3(nblocks), dim3(kBlock), 0, s, f, bc, k, V, uprev, partials);
    hipLaunchKernelGGL(diag_final_kernel<0>, dim3(1), dim3(64 * kDiag), 0, s, partials, nblocks, out);
}

template <typename T>
void launch_order_director(const Fields<T>& f, long c0, long n, double* order, double* director, hipStream_t s) {
    hipLaunchKernelGGL(order_director_kernel<T>, dim3(grid_for(n)), dim3(kBlock), 0, s, f, c0, n, order, director);
}

}  // namespace lbm
