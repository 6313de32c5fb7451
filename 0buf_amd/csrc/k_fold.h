/*
 * k_fold.h -- the periodic fold of the current (SetPeriodicCurrentComponent,
 * gpu_plasma.h:926-978) by classes of nodes, for the kernels that place a
 * step's arrivals (k_arrive.h, k_particles_f32.hip): the two stages touch
 * disjoint data and are both short, so one launch runs them, the fold in
 * workgroups behind the arrivals'.
 */
#ifndef K_FOLD_H
#define K_FOLD_H

#include "pic_internal.h"

template <typename JT>
struct FoldJ {
    JT *J[3];
};

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

/* the three k_fold_j launches x, y, z in one: thread t takes one class of
 * more than one node, folds its current in registers (x pairs, then y, then
 * z, as the launches run, with the same additions) and writes it back */
template <typename JT>
__device__ __forceinline__ void fold_class(const Grid &g, const FoldJ<JT> &f, unsigned t) {
    if (t >= shell_count(g)) return;
    const int Nx = g.Nx, Ny = g.Ny, Nz = g.Nz;
    int ri, rl, rk;
    const unsigned fx = 2u * Ny * Nz, fy = 2u * (unsigned)(Nx - 2) * Nz;
    if (t < fx) {                                    /* ri in {1, Nx} */
        const unsigned a = t / ((unsigned)Ny * Nz), r = t - a * ((unsigned)Ny * Nz);
        ri = a ? Nx : 1;
        rl = (int)(r / Nz) + 1;
        rk = (int)(r % Nz) + 1;
    } else if ((t -= fx) < fy) {                     /* rl in {1, Ny} */
        const unsigned a = t / ((unsigned)(Nx - 2) * Nz), r = t - a * ((unsigned)(Nx - 2) * Nz);
        rl = a ? Ny : 1;
        ri = (int)(r / Nz) + 2;
        rk = (int)(r % Nz) + 1;
    } else {                                         /* rk in {1, Nz} */
        t -= fy;
        const unsigned a = t / ((unsigned)(Nx - 2) * (Ny - 2)),
                       r = t - a * ((unsigned)(Nx - 2) * (Ny - 2));
        rk = a ? Nz : 1;
        ri = (int)(r / (Ny - 2)) + 2;
        rl = (int)(r % (Ny - 2)) + 2;
    }
    const unsigned sy = (unsigned)g.sy, sx = (unsigned)g.sx;
    const int px = ri == Nx ? 0 : ri == 1 ? Nx + 1 : -1;
    const int py = rl == Ny ? 0 : rl == 1 ? Ny + 1 : -1;
    const int pz = rk == Nz ? 0 : rk == 1 ? Nz + 1 : -1;
    const int X[2] = {ri, px}, Y[2] = {rl, py}, Z[2] = {rk, pz};
    auto member = [&](int s) {
        return ((s & 1) == 0 || px >= 0) && ((s & 2) == 0 || py >= 0) && ((s & 4) == 0 || pz >= 0);
    };
    unsigned m[8];
#pragma unroll
    for (int s = 0; s < 8; s++)
        m[s] = (unsigned)X[s & 1] * sx + (unsigned)Y[(s >> 1) & 1] * sy + (unsigned)Z[s >> 2];
    for (int cc = 0; cc < 3; cc++) {
        JT *J = f.J[cc];
        JT v[8];
#pragma unroll
        for (int s = 0; s < 8; s++) v[s] = member(s) ? J[m[s]] : (JT)0;
        if (px >= 0) {
#pragma unroll
            for (int s = 0; s < 8; s += 2)
                if (member(s)) fold_pair(v[s], v[s | 1], 0, cc, ri == Nx);
        }
        if (py >= 0) {
#pragma unroll
            for (int s = 0; s < 8; s++)
                if (!(s & 2) && member(s)) fold_pair(v[s], v[s | 2], 1, cc, rl == Ny);
        }
        if (pz >= 0) {
#pragma unroll
            for (int s = 0; s < 4; s++)
                if (member(s)) fold_pair(v[s], v[s | 4], 2, cc, rk == Nz);
        }
#pragma unroll
        for (int s = 0; s < 8; s++)
            if (member(s)) J[m[s]] = v[s];
    }
}

/* workgroups of PIC_BLOCK threads that fold every class */
inline unsigned fold_blocks(const Grid &g) {
    return (shell_count(g) + PIC_BLOCK - 1) / PIC_BLOCK;
}

#endif
