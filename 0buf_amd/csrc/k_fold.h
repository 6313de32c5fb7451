/*
 * k_fold.h -- the periodic fold of the current (SetPeriodicCurrentComponent,
 * gpu_plasma.h:926-978) by classes of nodes, for the kernels that place a
 * step's arrivals (k_arrive.h, k_particles_f32.hip): the two stages touch
 * disjoint data and are both short, so one launch runs them, the fold in
 * workgroups behind the arrivals'.
 */
#ifndef K_FOLD_H
#define K_FOLD_H

#include <type_traits>

#include "pic_internal.h"

/* fix (FP64 differentiable form, else null): the current still lies there as
 * int64 in units of 2^-48, to be converted on the way and cleared */
template <typename JT>
struct FoldJ {
    JT *J[3];
    long long *fix[3];
};

__device__ __forceinline__ double from_fixed(long long v) {
    return (double)v * (1.0 / PIC_J_SCALE64);
}

/* k_fold_j's four operations on one line, restricted to one partner pair:
 * r at the representative (position N or 1), p at its partner (0 or N+1),
 * for fold direction dir and current component cc:
 *   J[1] += J[N+1] (dir != cc);  J[N+1] = J[1] (unless dir = cc = y);
 *   J[0] += J[N];  J[N] = J[0]. */
template <typename JT>
__device__ __forceinline__ void fold_pair(JT &r, JT &p, int dir, int cc, bool at_n) {
    if (at_n) {
        const JT s = p + r;
        r = s;
        p = s;
    } else if (dir != cc) {
        const JT s = r + p;
        r = s;
        p = s;
    } else if (dir != 1) {
        p = r;
    }
}

/* the classes of nodes the current fold combines: along each axis the fold
 * only ever combines position N with 0 and position 1 with N+1 (N >= 3, so
 * the pairs are distinct), so the nodes whose coordinates are a
 * representative's own or its partner's (representative in [1,N]^3) form a
 * class no other class's fold touches.  The classes of more than one node
 * have their representative on a face of [1,N]^3: 2 Ny Nz with ri in
 * {1, Nx}, 2 (Nx-2) Nz with ri inside and rl in {1, Ny}, 2 (Nx-2)(Ny-2) with
 * ri, rl inside and rk in {1, Nz}. */
__host__ __device__ __forceinline__ unsigned shell_count(const Grid &g) {
    return 2u * (unsigned)g.Ny * g.Nz + 2u * (unsigned)(g.Nx - 2) * g.Nz +
           2u * (unsigned)(g.Nx - 2) * (g.Ny - 2);
}

/* class t: its representative (ri, rl, rk), the partner coordinate along each
 * axis (-1: none) and the node of member s (bit d of s: the partner's
 * coordinate along d) */
struct NodeClass {
    int ri, rl, rk, px, py, pz;
    unsigned m[8];
    __device__ __forceinline__ bool member(int s) const {
        return ((s & 1) == 0 || px >= 0) && ((s & 2) == 0 || py >= 0) && ((s & 4) == 0 || pz >= 0);
    }
    __device__ __forceinline__ int i(int s) const { return s & 1 ? px : ri; }
    __device__ __forceinline__ int l(int s) const { return s & 2 ? py : rl; }
    __device__ __forceinline__ int k(int s) const { return s & 4 ? pz : rk; }
};

__device__ __forceinline__ NodeClass node_class(const Grid &g, unsigned t) {
    const int Nx = g.Nx, Ny = g.Ny, Nz = g.Nz;
    NodeClass c;
    const unsigned fx = 2u * Ny * Nz, fy = 2u * (unsigned)(Nx - 2) * Nz;
    if (t < fx) {                                    /* ri in {1, Nx} */
        const unsigned a = t / ((unsigned)Ny * Nz), r = t - a * ((unsigned)Ny * Nz);
        c.ri = a ? Nx : 1;
        c.rl = (int)(r / Nz) + 1;
        c.rk = (int)(r % Nz) + 1;
    } else if ((t -= fx) < fy) {                     /* rl in {1, Ny} */
        const unsigned a = t / ((unsigned)(Nx - 2) * Nz), r = t - a * ((unsigned)(Nx - 2) * Nz);
        c.rl = a ? Ny : 1;
        c.ri = (int)(r / Nz) + 2;
        c.rk = (int)(r % Nz) + 1;
    } else {                                         /* rk in {1, Nz} */
        t -= fy;
        const unsigned a = t / ((unsigned)(Nx - 2) * (Ny - 2)),
                       r = t - a * ((unsigned)(Nx - 2) * (Ny - 2));
        c.rk = a ? Nz : 1;
        c.ri = (int)(r / (Ny - 2)) + 2;
        c.rl = (int)(r % (Ny - 2)) + 2;
    }
    c.px = c.ri == Nx ? 0 : c.ri == 1 ? Nx + 1 : -1;
    c.py = c.rl == Ny ? 0 : c.rl == 1 ? Ny + 1 : -1;
    c.pz = c.rk == Nz ? 0 : c.rk == 1 ? Nz + 1 : -1;
#pragma unroll
    for (int s = 0; s < 8; s++)
        c.m[s] = (unsigned)c.i(s) * (unsigned)g.sx + (unsigned)c.l(s) * (unsigned)g.sy +
                 (unsigned)c.k(s);
    return c;
}

/* the values of the three components at the class's nodes, op(component, v) on
 * each component's v[8] in registers, and back.  Every load is issued before
 * the first operation (a component after the other, each waited for memory on
 * its own: the arrival and fold of a small step 4.6 against 5.7 us, with the
 * conversion of a fixed-point current 8.6 against 11). */
template <typename JT, class Load, class Op>
__device__ __forceinline__ void on_class(const NodeClass &c, JT *const (&J)[3], Load load, Op op) {
    JT v[3][8];
#pragma unroll
    for (int cc = 0; cc < 3; cc++)
#pragma unroll
        for (int s = 0; s < 8; s++) v[cc][s] = c.member(s) ? load(cc, c.m[s]) : (JT)0;
#pragma unroll
    for (int cc = 0; cc < 3; cc++) op(cc, v[cc]);
#pragma unroll
    for (int cc = 0; cc < 3; cc++)
#pragma unroll
        for (int s = 0; s < 8; s++)
            if (c.member(s)) J[cc][c.m[s]] = v[cc][s];
}
template <typename JT, class Op>
__device__ __forceinline__ void on_class(const NodeClass &c, JT *const (&J)[3], Op op) {
    on_class(c, J, [&](int cc, unsigned m) { return J[cc][m]; }, op);
}

/* pair(v at the representative's side, v at the partner's, member s) over the
 * class's pairs along axis d (no pair: none) */
template <typename JT, class Pair>
__device__ __forceinline__ void class_pairs(const NodeClass &c, JT (&v)[8], int d, Pair pair) {
    if ((d == 0 ? c.px : d == 1 ? c.py : c.pz) < 0) return;
#pragma unroll
    for (int s = 0; s < 8; s++)
        if (!(s & (1 << d)) && c.member(s)) pair(v[s], v[s | (1 << d)], s);
}

/* the three k_fold_j launches x, y, z in one: thread t takes one class of
 * more than one node, folds its current in registers (x pairs, then y, then
 * z, as the launches run, with the same additions) and writes it back */
template <typename JT>
__device__ __forceinline__ void fold_class(const Grid &g, const FoldJ<JT> &f, unsigned t) {
    if (t >= shell_count(g)) return;
    const NodeClass c = node_class(g, t);
    const bool at_n[3] = {c.ri == g.Nx, c.rl == g.Ny, c.rk == g.Nz};
    auto fold = [&](int cc, JT (&v)[8]) {
#pragma unroll
        for (int d = 0; d < 3; d++)
            class_pairs(c, v, d, [&](JT &r, JT &p, int) { fold_pair(r, p, d, cc, at_n[d]); });
    };
    if constexpr (std::is_floating_point_v<JT>) {
        if (f.fix[0]) {
            on_class(c, f.J, [&](int cc, unsigned m) { return from_fixed(f.fix[cc][m]); }, fold);
            for (int cc = 0; cc < 3; cc++)
                for (int s = 0; s < 8; s++)
                    if (c.member(s)) f.fix[cc][c.m[s]] = 0;
            return;
        }
    }
    on_class(c, f.J, fold);
}

/* the nodes no class holds, node n: the conversion alone */
__device__ __forceinline__ void convert_inner(const Grid &g, const FoldJ<double> &f, unsigned n) {
    if (n >= (unsigned)g.G) return;
    const unsigned t = n / (unsigned)g.sy, k = n - t * (unsigned)g.sy;
    const unsigned i = t / (unsigned)(g.Ny + 2), l = t - i * (unsigned)(g.Ny + 2);
    if (i < 2 || (int)i >= g.Nx || l < 2 || (int)l >= g.Ny || k < 2 || (int)k >= g.Nz) return;
    long long v[3];
    for (int cc = 0; cc < 3; cc++) v[cc] = f.fix[cc][n];
    for (int cc = 0; cc < 3; cc++) {
        f.J[cc][n] = from_fixed(v[cc]);
        f.fix[cc][n] = 0;
    }
}

/* workgroups of PIC_BLOCK threads that fold every class */
inline unsigned fold_blocks(const Grid &g) {
    return (shell_count(g) + PIC_BLOCK - 1) / PIC_BLOCK;
}

#endif
