/*
 * k_particles_f64.hip -- particle stages of the FP64 plain form.
 *
 * One workgroup per tile of TX x TY x TZ cells:
 *   1. stage E and H^{n+1/2} of the tile's node box ((TX+2)(TY+2)(TZ+2)
 *      nodes: a cell's stencil reaches global nodes owner+0..owner+2) in LDS;
 *   2. each wavefront owns whole cells of the tile and walks their particles
 *      in flat order, in chunks of whole 128-byte line groups (consecutive
 *      lanes -> consecutive slots of a cell bucket, so loads coalesce and no
 *      line is shared by two chunks); a lane gathers, pushes, and deposits
 *      its charge-conserving current into an LDS copy of the tile's J box
 *      (ds_add_f64);
 *   3. the particle is wrapped, its fly direction and receiving cells are
 *      computed with the reference predicates; leavers go to the tile's
 *      departure region, stayers are compacted in place in flat order;
 *   4. the J box is added to the global arrays with FP64 atomics.
 * Decisions (cells, directions, receivers) mirror cell.h / particle.h in the
 * reference's evaluation order; the file is built with -ffp-contract=off and
 * writes the multiply-adds it wants fused as fma.
 *
 * Bound by vector issue (four fifths of its cycles), so what pays is fewer
 * instructions a particle: coordinates relative to the owner cell, one weight
 * factor per axis, fused segment weights, and every face test replaced by the
 * cell that the end lies in (k_receiver.h) took 20 steps at 256x64x64 cells,
 * 67M particles, from 68.0 to 60.6 ms, a step at 45x27x19 cells from 131 to
 * 118 us.
 */
#include <type_traits>

#include "k_arrive.h"
#include "k_tape.h"
#include "k_push_math.h"
#include "k_receiver.h"

#pragma clang fp contract(off)

namespace {

/* copies of the LDS J box, lane l depositing into copy l % JCOPIES: fewer
 * same-address conflicts of the LDS atomics (consecutive lanes hold
 * particles of one cell); the copies are summed in a fixed order before the
 * global flush */
#ifndef PIC_JCOPIES64
#define PIC_JCOPIES64 2
#endif

constexpr int TXC = 2, TYC = 4, TZC = 8;
constexpr int TXS = 2, TYS = 2, TZS = 4;   /* tiles of small boxes (make_tile_geom) */
constexpr int GS64 = 16;    /* slots of an FP64 array in one 128-byte line */
constexpr int JCOPIES = PIC_JCOPIES64;

struct PushArgs {
    Grid g;
    DivConst dc;
    TileGeom t;
    FieldPtrs f;
    PartPtrs p;
    QueuePtrs q;
    SpeciesTable sp;
    int dep_cap;
    DevStatus *st;
    DiffArgs d;        /* differentiable form (DIFF instantiation only) */
    int snap_on;
};

/* one node contribution a b to the LDS J box: FP64 atomic add, or in the
 * differentiable form the contribution (a scaled by 2^48) rounded to an integer
 * with the 1.5 2^52 shifter (exact for |a b| < 2^51) and added as int64 */
template <bool DIFF>
__device__ __forceinline__ void jadd(double *sJ, int n, double a, double b) {
    if constexpr (DIFF) {
        const double t = fma(a, b, 6755399441055744.0);
        const long long q = __double_as_longlong(t) - 0x4338000000000000LL;
        atomicAdd(reinterpret_cast<unsigned long long *>(sJ) + n, (unsigned long long)q);
    } else {
        atomicAdd(&sJ[n], a * b);
    }
}

/* cell.h:1511-1693 pqr: 12 node contributions of one straight segment a -> b
 * inside dual cell (ix, iy, iz), accumulated into the LDS J box at local node
 * (owner + tile index - 2).  Coordinates are relative to the owner cell's corner
 * (the reference's 1/2 (a + b) - h (i - 2.5) - x0 with x0 = 0); k = weight over
 * the face area and tau per axis, one factor where the reference multiplies by
 * the weight and divides by the product. */
template <int BY, int BZ, int JY0, int JZ0, bool DIFF>
__device__ __forceinline__ void pqr_lds(double *sJ, const Geo &c, const DivConst &dc, int ix,
                                        int iy, int iz, double ax, double ay, double az,
                                        double bx, double by, double bz, double kx, double ky,
                                        double kz, unsigned &bad, bool active) {
    if (!active) return;
    const int u = ix - 2, v = iy - 2, w = iz - 2;
    if ((unsigned)(u | v | w) > 1u) {
        bad = 1;
        return;
    }
    const double dx = fma(0.5, ax + bx, u ? -0.5 * c.hx : 0.5 * c.hx);
    const double dy = fma(0.5, ay + by, v ? -0.5 * c.hy : 0.5 * c.hy);
    const double dz = fma(0.5, az + bz, w ? -0.5 * c.hz : 0.5 * c.hz);
    const double dx1 = c.hx - dx, dy1 = c.hy - dy, dz1 = c.hz - dz;
    double su = bx - ax, sv = by - ay, sw = bz - az;
    const double su12 = su * dc.r12;
    const double s1 = (sv * dc.r12) * sw, s2 = su12 * sw, s3 = su12 * sv;
    su *= kx;
    sv *= ky;
    sw *= kz;
    const int n = c.n0 + (u ? BY * BZ : 0) + (v ? BZ : 0) + w;
    double *Jx = sJ, *Jy = sJ + JY0, *Jz = sJ + JZ0;
    const double wx0 = fma(dy1, dz1, s1), wx1 = fma(dy1, dz, -s1), wx2 = fma(dy, dz1, -s1),
                 wx3 = fma(dy, dz, s1);
    const double wy0 = fma(dx1, dz1, s2), wy1 = fma(dx1, dz, -s2), wy2 = fma(dx, dz1, -s2),
                 wy3 = fma(dx, dz, s2);
    const double wz0 = fma(dx1, dy1, s3), wz1 = fma(dx1, dy, -s3), wz2 = fma(dx, dy1, -s3),
                 wz3 = fma(dx, dy, s3);
    if constexpr (DIFF) {
        /* every contribution below 8 (2^51 units): the larger of each pair of
         * distances bounds the weights, wherever the segment lies (its end may
         * be many cells away at a large tau); where that bound does not tell,
         * the contributions themselves */
        const double mx = fmax(fabs(dx), fabs(dx1)), my = fmax(fabs(dy), fabs(dy1)),
                     mz = fmax(fabs(dz), fabs(dz1));
        if (!(fabs(su) * fma(my, mz, fabs(s1)) < 7.9 && fabs(sv) * fma(mx, mz, fabs(s2)) < 7.9 &&
              fabs(sw) * fma(mx, my, fabs(s3)) < 7.9)) {
            auto over = [](double a, double w0, double w1, double w2, double w3) {
                return !(fabs(a * w0) < 8.0 && fabs(a * w1) < 8.0 && fabs(a * w2) < 8.0 &&
                         fabs(a * w3) < 8.0);
            };
            if (over(su, wx0, wx1, wx2, wx3) || over(sv, wy0, wy1, wy2, wy3) ||
                over(sw, wz0, wz1, wz2, wz3))
                bad = 1;
        }
        su *= PIC_J_SCALE64;
        sv *= PIC_J_SCALE64;
        sw *= PIC_J_SCALE64;
    }
    jadd<DIFF>(Jx, n, su, wx0);
    jadd<DIFF>(Jx, n + 1, su, wx1);
    jadd<DIFF>(Jx, n + BZ, su, wx2);
    jadd<DIFF>(Jx, n + BZ + 1, su, wx3);
    jadd<DIFF>(Jy, n, sv, wy0);
    jadd<DIFF>(Jy, n + 1, sv, wy1);
    jadd<DIFF>(Jy, n + BY * BZ, sv, wy2);
    jadd<DIFF>(Jy, n + BY * BZ + 1, sv, wy3);
    jadd<DIFF>(Jz, n, sw, wz0);
    jadd<DIFF>(Jz, n + BZ, sw, wz1);
    jadd<DIFF>(Jz, n + BY * BZ, sw, wz2);
    jadd<DIFF>(Jz, n + BY * BZ + BZ, sw, wz3);
}

/* flyDirection (cell.h:694-701) along one axis: 0, 1, 2 */
__device__ __forceinline__ int flies(double v, double v0, double h, int i, int n, double L) {
    return ((v > v0 + h) && (v < v0 + 2 * h)) || ((v < h) && (i == n - 1))
               ? 2
               : ((v < v0) || ((v > L - h) && (i == 0)) ? 0 : 1);
}

/* 4 waves per SIMD (at most 128 VGPRs): the FP64 chains of the push are
 * latency-bound at 3 */
template <int TX, int TY, int TZ, bool DIFF, bool TAPE, int NT>
__global__ __launch_bounds__(NT, 4) void k_push_deposit(PushArgs a) {
    constexpr int C = TX * TY * TZ;
    constexpr int BX = TX + 2, BY = TY + 2, BZ = TZ + 2, NB = BX * BY * BZ;
    /* the current box: Jx (dual along x) takes x planes 0..TX only, Jy and Jz
     * all of them; copies JS apart, 8 mod 16 doubles, so that the two copies'
     * nodes of a cell lie on other banks */
    constexpr int NBX = (TX + 1) * BY * BZ;
    constexpr int JY0 = NBX, JZ0 = NBX + NB, NJ = NBX + 2 * NB, JS = (NJ + 15) / 16 * 16 + 8;
    /* field boxes; the differentiable form keeps (value, difference to the
     * next node along z) */
    using Node = std::conditional_t<DIFF, double2, double>;
    __shared__ Node sF[6 * NB];
    __shared__ double sJ[JCOPIES * JS];
    __shared__ int sOff[C + 1];
    __shared__ int sCnt[C];
    __shared__ int sLeave[C];
    __shared__ int sOut[C];
    __shared__ int sBase[C];     /* first slot of each cell, relative to the tile's first cell */
    __shared__ int sG[C + 1];    /* first line group of each cell */
    __shared__ int sQ;
    __shared__ unsigned sFlags;
    __shared__ unsigned long long sDrop, sDup;
    __shared__ double sSpec[PIC_MAX_SLOTS][4];   /* q/m tau/2 and m over Dx, Dy, Dz per species slot */
    extern __shared__ unsigned sGrp[];    /* line groups of the tile */
    double *const myJ = sJ + (threadIdx.x % JCOPIES) * JS;

    const Grid &g = a.g;
    const int tid = threadIdx.x;
    const bool snap = DIFF && a.snap_on;

    const TileAt at = tile_of_block(a.t, blockIdx.x);
    const long tile = at.tile;
    const int tx = at.tx, ty = at.ty, tz = at.tz;
    /* workgroup-uniform (the divisions run on the vector unit; readfirstlane
     * keeps the tile's base addresses scalar) */
    const int I0 = __builtin_amdgcn_readfirstlane(tx * TX);
    const int L0 = __builtin_amdgcn_readfirstlane(ty * TY);
    const int K0 = __builtin_amdgcn_readfirstlane(tz * TZ);
    const int cap = a.p.cap;

    /* Thread n takes box node n of the six field boxes (one decode, one
     * 32-bit offset: the grid has fewer than 2^31 nodes) and cell n of the
     * tile; every global load is issued before the first LDS write. */
    static_assert(NB <= NT && C <= NT, "one box node and one cell per thread");
    const int nu = tid / (BY * BZ), nv = (tid / BZ) % BY, nw = tid % BZ;
    const bool node_in = tid < NB && I0 + nu <= g.Nx + 1 && L0 + nv <= g.Ny + 1 &&
                         K0 + nw <= g.Nz + 1;
    const unsigned noff = (unsigned)(I0 + nu) * g.sx + (unsigned)(L0 + nv) * g.sy + (K0 + nw);
    {
        double fv[6], fd[6];   /* node value, next node's value (0 outside the grid) */
#pragma unroll
        for (int q = 0; q < 6; q++) fv[q] = fd[q] = 0.0;
        if (node_in) {
#pragma unroll
            for (int q = 0; q < 6; q++) fv[q] = a.f.f[PIC_EX + q][noff];
        }
        if (DIFF && node_in && nw + 1 < BZ && K0 + nw + 1 <= g.Nz + 1) {
#pragma unroll
            for (int q = 0; q < 6; q++) fd[q] = a.f.f[PIC_EX + q][noff + 1];
        }
        const int ca = tid / (TY * TZ), cb = (tid / TZ) % TY, cc = tid % TZ;
        const int gi = I0 + ca, gl = L0 + cb, gk = K0 + cc;
        int cnt = 0;
        if (tid < C && gi < g.Nx && gl < g.Ny && gk < g.Nz) {
            const long cell = ((long)gi * g.Ny + gl) * g.Nz + gk;
            cnt = a.p.count[cell];
            cnt = cnt < cap ? cnt : cap;
            if (snap) a.d.snap.count[cell] = cnt;
        }
        if (tid < NB) {
#pragma unroll
            for (int q = 0; q < 6; q++) {
                if constexpr (DIFF) sF[q * NB + tid] = make_double2(fv[q], fd[q] - fv[q]);
                else sF[q * NB + tid] = fv[q];
            }
        }
        if (tid < C) {
            sCnt[tid] = cnt;
            sLeave[tid] = 0;
            sOut[tid] = 0;
            sBase[tid] = ((ca * g.Ny + cb) * g.Nz + cc) * cap;
        }
    }
    for (int e = tid; e < JCOPIES * JS; e += NT) sJ[e] = 0.0;
    /* the factors of each species slot: a kernel-argument table indexed by a
     * per-particle value would be a vector memory load in the loop, whose
     * wait would also wait for the particle loads in flight */
    if (tid < PIC_MAX_SLOTS) {
        sSpec[tid][0] = a.sp.q_m[tid] * g.tau * 0.5;
        sSpec[tid][1] = a.sp.m[tid] / a.dc.Dx;
        sSpec[tid][2] = a.sp.m[tid] / a.dc.Dy;
        sSpec[tid][3] = a.sp.m[tid] / a.dc.Dz;
    }
    if (tid == 0) {
        sQ = 0;
        sFlags = 0;
        sDrop = 0;
        sDup = 0;
    }
    __syncthreads();
    static_assert(C <= 64, "one wavefront scans the tile's cells");
    if (tid < 64) {   /* first particle and first line group of each cell */
        const int cnt = tid < C ? sCnt[tid] : 0;
        int tot_s, tot_g;
        const int so = wave_excl_scan(cnt, tot_s),
                  sg = wave_excl_scan((cnt + GS64 - 1) / GS64, tot_g);
        if (tid < C) {
            sOff[tid] = so;
            sG[tid] = sg;
        }
        if (tid == 0) {
            sOff[C] = tot_s;
            sG[C] = tot_g;
        }
    }
    __syncthreads();
    build_groups<TX, TY, TZ, GS64>(sCnt, sG, sGrp, tid, NT);
    __syncthreads();

    /* per-tile bases of the particle arrays: slot rel of the tile is
     * cell-bucket slot pbase + rel */
    const long pbase = (((long)I0 * g.Ny + L0) * g.Nz + K0) * cap;
    double *const P0 = a.p.p[0] + pbase, *const P1 = a.p.p[1] + pbase,
                  *const P2 = a.p.p[2] + pbase, *const P3 = a.p.p[3] + pbase,
                  *const P4 = a.p.p[4] + pbase, *const P5 = a.p.p[5] + pbase;
    unsigned char *const SP = a.p.sp + pbase;
    int *const ID = DIFF ? a.p.id + pbase : nullptr;
    Leaver64 *const QT = a.q.e + tile * (long)a.q.qcap;   /* the tile's departure queue */

    /* where the tile's record starts and how many of its particles have room
     * there, read before the loop: a load in it waits for every one before */
    const long snap0 = snap ? uniform(a.d.snap_off[tile]) : 0;
    const unsigned snap_n = record_room(snap, snap0, a.d.snap_room);

    const double hx = g.hx, hy = g.hy, hz = g.hz, tau = g.tau;
    unsigned bad = 0;
    /* each wavefront owns whole cells and walks their particles in chunks of
     * 64 consecutive ones (a line group may be split between two consecutive
     * chunks); stayers are compacted in place in flat order */
    const int lane = tid & 63, wv = tid >> 6;
    const int ghi = __builtin_amdgcn_readfirstlane(
        sG[wave_first_cell<C>(sOff, wv + 1, NT / 64)]);
    int g0 = __builtin_amdgcn_readfirstlane(sG[wave_first_cell<C>(sOff, wv, NT / 64)]);
    int o0 = 0;
    int carry_cell = -1, carry_cnt = 0;
    while (g0 < ghi) {
        unsigned long long starts = 0, runs = 0;
        int lanes = 0, onext = 0;
        const int gnext = compose_full_chunk(sGrp, g0, o0, ghi, starts, lanes, runs, onext);
        const bool valid = lane < lanes;
        int c = 0, j = 0;
        bool stays = false;
        double xn = 0, yn = 0, zn = 0, pu = 0, pv = 0, pw = 0;
        unsigned char s = 0;
        int pid = 0;
        tape_word tout = 0;    /* this step's decisions (decision tape, record mode) */
        if (valid) {
            const unsigned long long msk = starts & (~0ull >> (63 - lane));
            const int gidx = __popcll(msk) - 1;
            const unsigned ge = sGrp[g0 + gidx];
            c = group_cell(ge);
            j = group_start(ge) + (lane - (63 - __clzll(msk))) + (gidx == 0 ? o0 : 0);
            const unsigned rel = (unsigned)(sBase[c] + j);
            const int ca = c / (TY * TZ), cb = (c / TZ) % TY, cc = c % TZ;
            const int gi = I0 + ca, gl = L0 + cb, gk = K0 + cc;
            Geo G;
            G.n0 = (int)__umul24(__umul24((unsigned)ca, BY) + (unsigned)cb, BZ) + cc;
            G.hx = hx; G.hy = hy; G.hz = hz;
            const double x0 = (double)gi * hx, y0 = (double)gl * hy, z0 = (double)gk * hz;

            const double x = slot(P0, rel), y = slot(P1, rel), z = slot(P2, rel);
            pu = slot(P3, rel);
            pv = slot(P4, rel);
            pw = slot(P5, rel);
            s = slot(SP, rel);
            pid = DIFF ? slot(ID, rel) : 0;
            /* decision tape (differentiable form): record this step's
             * decisions, or replay a recorded run's */
            const bool trec = TAPE && a.d.tape_mode == PIC_TAPE_RECORD;
            const bool trep = TAPE && a.d.tape_mode == PIC_TAPE_REPLAY;
            const bool tin = (trec || trep) && pid >= 0 && pid < a.d.tape_n;
            tape_word tw = 0;
            if (trep) {
                if (tin) tw = a.d.tape_row[pid];
                if (!tin || !((tw >> TAPE_VALID) & 1ull) || ((tw >> TAPE_BAD) & 1ull)) bad = 1;
            }
            const unsigned r = (unsigned)(sOff[c] + j);
            if (r < snap_n) {
                slot(a.d.snap.p[0] + snap0, r) = x;
                slot(a.d.snap.p[1] + snap0, r) = y;
                slot(a.d.snap.p[2] + snap0, r) = z;
                slot(a.d.snap.p[3] + snap0, r) = pu;
                slot(a.d.snap.p[4] + snap0, r) = pv;
                slot(a.d.snap.p[5] + snap0, r) = pw;
                slot(a.d.snap.sp + snap0, r) = s;
                slot(a.d.snap.id + snap0, r) = pid;
            }

            /* relative to the owner cell's corner */
            const double xl = x - x0, yl = y - y0, zl = z - z0;
            const double frx = divc(xl, hx, a.dc.rhx);
            const double fry = divc(yl, hy, a.dc.rhy);
            const double frz = divc(zl, hz, a.dc.rhz);
            double Ex = 0, Ey = 0, Ez = 0, Hx = 0, Hy = 0, Hz = 0;
            const bool neg = trep ? (tw & 1ull) != 0 : (x < 0 || y < 0 || z < 0);
            if (trec && neg) tout |= 1ull;
            if (!neg) {
                GatherIdx W = gather_index(x, y, z, frx, fry, frz, g, a.dc);
                const int gc[3] = {gi, gl, gk};
                if (trep) {
                    int *ii[6] = {&W.ix, &W.i1x, &W.iy, &W.i1y, &W.iz, &W.i1z};
                    for (int q = 0; q < 6; q++) *ii[q] = tape_get(tw, TAPE_GIDX + q, 1, 2);
                    for (int d = 0; d < 3; d++) {
                        W.f1[d] = gc[d] + tape_get(tw, TAPE_FLOOR + 4 * d, 2, 0);
                        W.f15[d] = gc[d] + tape_get(tw, TAPE_FLOOR + 4 * d + 2, 2, 0);
                    }
                    gather_weights(W, divc(x, g.hx, a.dc.rhx), divc(y, g.hy, a.dc.rhy),
                                   divc(z, g.hz, a.dc.rhz));
                    W.ok = gather_ok(W);
                }
                if (trec) {
                    const int ii[6] = {W.ix, W.i1x, W.iy, W.i1y, W.iz, W.i1z};
                    for (int q = 0; q < 6; q++) tape_put(tout, TAPE_GIDX + q, 1, ii[q], 2);
                    for (int d = 0; d < 3; d++) {
                        tape_put(tout, TAPE_FLOOR + 4 * d, 2, (int)W.f1[d] - gc[d], 0);
                        tape_put(tout, TAPE_FLOOR + 4 * d + 2, 2, (int)W.f15[d] - gc[d], 0);
                    }
                }
                const double s1 = W.s1, s2 = W.s2, s3 = W.s3, s4 = W.s4, s5 = W.s5, s6 = W.s6;
                const double s11 = 1. - W.s1, s21 = 1. - W.s2, s31 = 1. - W.s3, s41 = 1. - W.s4,
                             s51 = 1. - W.s5, s61 = 1. - W.s6;
                if (!W.ok) {
                    bad = 1;
                } else {
                    const int X = G.n0 + (W.ix != 2 ? BY * BZ : 0),
                              X1 = G.n0 + (W.i1x != 2 ? BY * BZ : 0),
                              Y = W.iy != 2 ? BZ : 0, Y1 = W.i1y != 2 ? BZ : 0, Z = W.iz - 2,
                              Z1 = W.i1z - 2;
                    Ex = interp<BY, BZ>(sF + 0 * NB, X + Y1 + Z1, s11, s41, s61, s1, s4, s6);
                    Ey = interp<BY, BZ>(sF + 1 * NB, X1 + Y + Z1, s21, s31, s61, s2, s3, s6);
                    Ez = interp<BY, BZ>(sF + 2 * NB, X1 + Y1 + Z, s21, s41, s51, s2, s4, s5);
                    Hx = interp<BY, BZ>(sF + 3 * NB, X1 + Y + Z, s21, s31, s51, s2, s3, s5);
                    Hy = interp<BY, BZ>(sF + 4 * NB, X + Y1 + Z, s11, s41, s51, s1, s4, s5);
                    Hz = interp<BY, BZ>(sF + 5 * NB, X + Y + Z1, s11, s31, s61, s1, s3, s6);
                }
            }

            /* Particle::Move (particle.h:160-202) */
            const Boris B = boris_move<DIFF>(pu, pv, pw, Ex, Ey, Ez, Hx, Hy, Hz, sSpec[s][0]);
            pu = B.p1[0];
            pv = B.p1[1];
            pw = B.p1[2];
            const double x1 = advance<DIFF>(x, tau, B.g2, pu), y1 = advance<DIFF>(y, tau, B.g2, pv),
                         z1 = advance<DIFF>(z, tau, B.g2, pw);
            const double x1l = x1 - x0, y1l = y1 - y0, z1l = z1 - z0;
            const double t1x = divc(x1l, hx, a.dc.rhx), t1y = divc(y1l, hy, a.dc.rhy),
                         t1z = divc(z1l, hz, a.dc.rhz);

            /* CurrentToMesh (cell.h:1306-1422): one code path for every lane;
             * without a crossing the first segment is the whole path (x2 = x1)
             * and the second is skipped */
            {
                const Relay R =
                    trep ? relay_from(xl, yl, zl, x1l, y1l, z1l, G, tape_get(tw, TAPE_RI1, 1, 2),
                                      tape_get(tw, TAPE_RI1 + 1, 1, 2),
                                      tape_get(tw, TAPE_RI1 + 2, 1, 2),
                                      tape_get(tw, TAPE_RI2, 2, 1), tape_get(tw, TAPE_RI2 + 2, 2, 1),
                                      tape_get(tw, TAPE_RI2 + 4, 2, 1))
                         : relay_point(xl, yl, zl, x1l, y1l, z1l, frx, fry, frz, t1x, t1y, t1z, G);
                if (trec) {
                    tape_put(tout, TAPE_RI1, 1, R.i1x, 2);
                    tape_put(tout, TAPE_RI1 + 1, 1, R.i1y, 2);
                    tape_put(tout, TAPE_RI1 + 2, 1, R.i1z, 2);
                    tape_put(tout, TAPE_RI2, 2, R.i2x, 1);
                    tape_put(tout, TAPE_RI2 + 2, 2, R.i2y, 1);
                    tape_put(tout, TAPE_RI2 + 4, 2, R.i2z, 1);
                }
                const int m = R.m;
                const double e1x = m ? R.x2x : x1l, e1y = m ? R.x2y : y1l, e1z = m ? R.x2z : z1l;
                const double kx = sSpec[s][1], ky = sSpec[s][2], kz = sSpec[s][3];
                pqr_lds<BY, BZ, JY0, JZ0, DIFF>(myJ, G, a.dc, R.i1x, R.i1y, R.i1z, xl, yl, zl, e1x,
                                                e1y, e1z, kx, ky, kz, bad, true);
                /* (kept waiting in registers until a lane has a second one, as
                 * the FP32 push does, they spill at 128 VGPRs: 2.47 against
                 * 2.38 ms at 67M particles) */
                pqr_lds<BY, BZ, JY0, JZ0, DIFF>(myJ, G, a.dc, R.i2x, R.i2y, R.i2z, R.x2x, R.x2y,
                                                R.x2z, x1l, y1l, z1l, kx, ky, kz, bad, m != 0);
            }

            /* x <- x1, Reflect (cell.h:1410-1478), flyDirection (cell.h:694-701) with
             * the owner cell's geometry, the test of the own cell, and the
             * receivers: GPU_ArrangeFlights (kernels.cu:316-370) gives every bulk
             * cell of the 27-neighbourhood (getWrapCellNumber) whose isPointInCell
             * (cell.h:717) holds a copy; per axis the test is separable, so the
             * receivers are a product of per-axis sets, bit d+1 set when
             * neighbour d in {-1,0,1} accepts.  All follow from the cell that x1
             * lies in; the tests themselves only where some lane lies near a face
             * (axis_step), and for the decision tape. */
            int dx = 0, dy = 0, dz = 0;
            bool near = TAPE;
            if (!TAPE) {
                xn = axis_step(x1, t1x, gi, g.Nx, g.Lx, dx, near);
                yn = axis_step(y1, t1y, gl, g.Ny, g.Ly, dy, near);
                zn = axis_step(z1, t1z, gk, g.Nz, g.Lz, dz, near);
            }
            stays = (dx | dy | dz) == 0;
            bool inside = stays;
            unsigned bx = 1u << (dx + 1), by = 1u << (dy + 1), bz = 1u << (dz + 1);
            if (near) {
                if (TAPE && (trec || trep)) {
                    const double v1[3] = {x1, y1, z1}, Lm[3] = {g.Lx, g.Ly, g.Lz};
                    double vn[3];
                    for (int d = 0; d < 3; d++) {
                        const int k = trep ? tape_get(tw, TAPE_REFL + 2 * d, 2, 0)
                                           : reflect_case(v1[d], Lm[d]);
                        if (trec) tape_put(tout, TAPE_REFL + 2 * d, 2, k, 0);
                        vn[d] = reflect_apply(v1[d], Lm[d], k);
                    }
                    xn = vn[0];
                    yn = vn[1];
                    zn = vn[2];
                } else {
                    xn = reflect1(x1, g.Lx);
                    yn = reflect1(y1, g.Ly);
                    zn = reflect1(z1, g.Lz);
                }
                stays = flies(xn, x0, hx, gi, g.Nx, g.Lx) == 1 &&
                        flies(yn, y0, hy, gl, g.Ny, g.Ly) == 1 &&
                        flies(zn, z0, hz, gk, g.Nz, g.Lz) == 1;
                inside = (x0 <= xn) && (xn < x0 + hx) && (y0 <= yn) && (yn < y0 + hy) &&
                         (z0 <= zn) && (zn < z0 + hz);
                if (!stays || TAPE) {
                    bx = receivers(xn, hx, gi, g.Nx);
                    by = receivers(yn, hy, gl, g.Ny);
                    bz = receivers(zn, hz, gk, g.Nz);
                }
            }
            if (!inside) atomicAdd(&sOut[c], 1);

            /* a replayed word that cannot be trusted keeps its particle in
             * place (the step reports PIC_F_RANGE) */
            if (trep) stays = ((tw >> TAPE_STAY) & 1ull) || !tin ||
                              !((tw >> TAPE_VALID) & 1ull) || ((tw >> TAPE_BAD) & 1ull);
            if (trec && stays) tout |= 1ull << TAPE_STAY;
            if (!stays) {
                atomicAdd(&sLeave[c], 1);
                if (trec) {
                    const unsigned bb[3] = {bx, by, bz};
                    for (int d = 0; d < 3; d++) {
                        if (__popc(bb[d]) == 1) tape_put(tout, TAPE_RECV + 2 * d, 2, __ffs(bb[d]) - 1, 0);
                        else tout |= 1ull << TAPE_BAD;
                    }
                }
                if (trep) {
                    /* the recorded receiver, one per axis (0..2) */
                    unsigned *bb[3] = {&bx, &by, &bz};
                    for (int d = 0; d < 3; d++) {
                        const int k = tape_get(tw, TAPE_RECV + 2 * d, 2, 0);
                        if (k > 2) bad = 1;
                        *bb[d] = k > 2 ? 0u : 1u << k;
                    }
                }
                const int ncopy = __popc(bx) * __popc(by) * __popc(bz);
                if (ncopy == 0) atomicAdd(&sDrop, 1ull);
                if (ncopy > 1) atomicAdd(&sDup, (unsigned long long)(ncopy - 1));
                if (ncopy > 0) {
                    const int first = atomicAdd(&sQ, ncopy);
                    /* the record of receiver (ax, ay, az): axis offsets 0..2 */
                    auto queue = [&](int ax, int ay, int az, int idx) {
                        if (idx >= a.q.qcap) return;
                        int rx = gi + ax - 1, ry = gl + ay - 1, rz = gk + az - 1;
                        if (rx >= g.Nx) rx -= g.Nx; else if (rx < 0) rx += g.Nx;
                        if (ry >= g.Ny) ry -= g.Ny; else if (ry < 0) ry += g.Ny;
                        if (rz >= g.Nz) rz -= g.Nz; else if (rz < 0) rz += g.Nz;
                        const int h = G.n0 + (int)__umul24((unsigned)ax, BY * BZ) +
                                      (int)__umul24((unsigned)ay, BZ) + az;
                        Leaver64 &e = slot(QT, (unsigned)idx);
                        e.xy = make_double2(xn, yn);
                        e.zu = make_double2(zn, pu);
                        e.vw = make_double2(pv, pw);
                        *(int4 *)&e.dest =
                            make_int4((rx * g.Ny + ry) * g.Nz + rz, (int)s | h << 8, pid, -1);
                    };
                    /* nearly every leaver has one receiver: the lanes write
                     * theirs together.  (As a loop over the 27 neighbours,
                     * unrolled, the wavefront ran the stores once for every
                     * neighbour some lane goes to.) */
                    const int ax0 = __ffs(bx) - 1, ay0 = __ffs(by) - 1, az0 = __ffs(bz) - 1;
                    queue(ax0, ay0, az0, first);
                    if (ncopy > 1) {
                        /* a one-ulp overlap of cells: the others, in the
                         * reference's scan order (x, then y, then z) */
                        int kq = 0;
#pragma unroll 1
                        for (int k = 0; k < 27; k++) {
                            const int ax = k / 9, ay = (k / 3) % 3, az = k % 3;
                            if (!((bx >> ax) & (by >> ay) & (bz >> az) & 1u)) continue;
                            if (kq > 0) queue(ax, ay, az, first + kq);
                            kq++;
                        }
                    }
                }
            }
        }

        if constexpr (TAPE) {
            if (valid && a.d.tape_mode == PIC_TAPE_RECORD && pid >= 0 && pid < a.d.tape_n)
                a.d.tape_row[pid] = tout | (1ull << TAPE_VALID);
        }

        /* stayers compacted in flat order (the reference removes leavers by
         * swap-with-last, removeParticleFromSurfaceDevice, cell.h:391-432;
         * the order inside a cell changes no result but the rounding of the
         * FP64 atomic sums, which have no fixed order either) */
        const int rank = stable_rank_runs(runs, c, valid, stays, carry_cell, carry_cnt);
        if (valid && stays) {
            const unsigned dst = (unsigned)(sBase[c] + rank);
            slot(P0, dst) = xn;
            slot(P1, dst) = yn;
            slot(P2, dst) = zn;
            slot(P3, dst) = pu;
            slot(P4, dst) = pv;
            slot(P5, dst) = pw;
            if (rank != j) {
                slot(SP, dst) = s;
                if (DIFF) slot(ID, dst) = pid;
            }
        }
        g0 = gnext;
        o0 = onext;
    }
    if (bad) atomicOr(&sFlags, (unsigned)PIC_F_RANGE);
    __syncthreads();

    int maxout = 0;
    for (int c = tid; c < C; c += NT) {
        const int ca = c / (TY * TZ), cb = (c / TZ) % TY, cc = c % TZ;
        const int gi = I0 + ca, gl = L0 + cb, gk = K0 + cc;
        if (gi >= g.Nx || gl >= g.Ny || gk >= g.Nz) continue;
        const long cell = ((long)gi * g.Ny + gl) * g.Nz + gk;
        a.p.count[cell] = sCnt[c] - sLeave[c];
        if (sOut[c] > maxout) maxout = sOut[c];
    }

    /* tile J box -> global J (GPU_WriteAllCurrents, kernels.cu:83-112) */
    if (tid < NB) {   /* thread n adds box node n of the three components */
#pragma unroll
        for (int comp = 0; comp < 3; comp++) {
            constexpr int J0[3] = {0, JY0, JZ0};
            if (comp == 0 && tid >= NBX) continue;
            const int e = J0[comp] + tid;
            if constexpr (DIFF) {
                const unsigned long long *u = reinterpret_cast<const unsigned long long *>(sJ);
                unsigned long long val = u[e];
                for (int r = 1; r < JCOPIES; r++) val += u[r * JS + e];
                if (val != 0ull && node_in)
                    atomicAdd(reinterpret_cast<unsigned long long *>(a.d.jfix[comp]) + noff, val);
            } else {
                double val = sJ[e];
                for (int r = 1; r < JCOPIES; r++) val += sJ[r * JS + e];
                if (val != 0.0 && node_in) atomicAdd(&a.f.f[PIC_JX + comp][noff], val);
            }
        }
    }

    if (maxout > 0) {
        if (a.dep_cap > 0 && maxout > a.dep_cap) atomicOr(&sFlags, (unsigned)PIC_F_TOO_MANY);
        if (maxout > a.st->max_dep) atomicMax(&a.st->max_dep, maxout);
    }
    __syncthreads();
    if (tid == 0) {
        int nq = sQ;
        if (nq > a.q.qcap) {
            atomicOr(&sFlags, (unsigned)PIC_F_QUEUE_OVERFLOW);
            nq = a.q.qcap;
        }
        a.q.count[tile] = nq;
        if (sFlags) atomicOr(&a.st->flags, sFlags);
        if (sDrop) atomicAdd(&a.st->dropped, sDrop);
        if (sDup) atomicAdd(&a.st->duplicated, sDup);
    }
}

/* differentiable form: fixed-point J -> the FP64 J arrays (exact for
 * |J| < 2^5), and the fixed-point arrays cleared for the next step */
__global__ __launch_bounds__(PIC_BLOCK) void k_jfix_to_f64(long G, FieldPtrs f, DiffArgs d) {
    const long n = (long)blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (n >= G) return;
    for (int c = 0; c < 3; c++) {
        const long long v = d.jfix[c][n];
        f.f[PIC_JX + c][n] = (double)v * (1.0 / PIC_J_SCALE64);
        d.jfix[c][n] = 0;
    }
}


/* initial upload: compact cell-sorted arrays -> buckets */
__global__ __launch_bounds__(PIC_BLOCK) void k_scatter_load(const long *off, long ncell,
                                                           const double *s0, const double *s1,
                                                           const double *s2, const double *s3,
                                                           const double *s4, const double *s5,
                                                           const unsigned char *ssp, PartPtrs p) {
    const long c = group_cell_index();
    if (c >= ncell) return;
    const long first = off[c], n = off[c + 1] - first;
    if (threadIdx.x % CELL_LANES == 0) p.count[c] = (int)n;
    for (int j = threadIdx.x % CELL_LANES; j < n && j < p.cap; j += CELL_LANES) {
        const long e = c * p.cap + j, src = first + j;
        p.p[0][e] = s0[src];
        p.p[1][e] = s1[src];
        p.p[2][e] = s2[src];
        p.p[3][e] = s3[src];
        p.p[4][e] = s4[src];
        p.p[5][e] = s5[src];
        p.sp[e] = ssp[src];
    }
}

__global__ __launch_bounds__(PIC_BLOCK) void k_repack(long ncell, PartPtrs from, PartPtrs to) {
    const long e = (long)blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (e >= ncell * from.cap) return;
    const long c = e / from.cap;
    const int j = (int)(e % from.cap);
    int n = from.count[c];
    if (n > from.cap) n = from.cap;
    if (j >= n) return;
    const long dst = c * to.cap + j;
    for (int k = 0; k < 6; k++) to.p[k][dst] = from.p[k][e];
    to.sp[dst] = from.sp[e];
    if (to.id) to.id[dst] = from.id[e];
}

__global__ __launch_bounds__(PIC_BLOCK) void k_scatter_ids(const long *off, long ncell,
                                                          const int *src, PartPtrs p) {
    const long c = group_cell_index();
    if (c >= ncell) return;
    const long first = off[c], n = off[c + 1] - first;
    for (int j = threadIdx.x % CELL_LANES; j < n && j < p.cap; j += CELL_LANES)
        p.id[c * p.cap + j] = src[first + j];
}

__global__ __launch_bounds__(PIC_BLOCK) void k_fix_arrivals(QueuePtrs q, int oldcap, PartPtrs to) {
    const long tile = blockIdx.x;
    const int n = q.count[tile];
    const Leaver64 *const Q = q.e + tile * (long)q.qcap;
    for (int j = threadIdx.x; j < n; j += PIC_BLOCK) {
        const int slot = Q[j].slot;
        if (slot < oldcap || slot >= to.cap) continue;
        const Leaver64 r = Q[j];
        const long dst = (long)r.dest * to.cap + slot;
        to.p[0][dst] = r.xy.x;
        to.p[1][dst] = r.xy.y;
        to.p[2][dst] = r.zu.x;
        to.p[3][dst] = r.zu.y;
        to.p[4][dst] = r.vw.x;
        to.p[5][dst] = r.vw.y;
        to.sp[dst] = (unsigned char)(r.where & 255);
        if (to.id) to.id[dst] = r.id;
    }
}

__global__ __launch_bounds__(PIC_BLOCK) void k_gather_particles(long ncell, const long *off,
                                                               PartPtrs p, double *d0, double *d1,
                                                               double *d2, double *d3, double *d4,
                                                               double *d5, unsigned char *dsp,
                                                               int *dcell, int *did) {
    const long c = group_cell_index();
    if (c >= ncell) return;
    const long first = off[c], n = off[c + 1] - first;
    for (int j = threadIdx.x % CELL_LANES; j < n && j < p.cap; j += CELL_LANES) {
        const long e = c * p.cap + j, dst = first + j;
        d0[dst] = p.p[0][e];
        d1[dst] = p.p[1][e];
        d2[dst] = p.p[2][e];
        d3[dst] = p.p[3][e];
        d4[dst] = p.p[4][e];
        d5[dst] = p.p[5][e];
        dsp[dst] = p.sp[e];
        if (dcell) dcell[dst] = (int)c;
        if (did) did[dst] = p.id ? p.id[e] : -1;
    }
}

inline unsigned blocks_for(long n) { return (unsigned)((n + PIC_BLOCK - 1) / PIC_BLOCK); }

}  // namespace


void launch_push_deposit_f64(const Grid &g, const TileGeom &t, FieldPtrs f, PartPtrs p,
                             QueuePtrs q, SpeciesTable sp, int dep_cap, DevStatus *st,
                             const DiffArgs *diff, hipStream_t s) {
    PushArgs a;
    a.g = g;
    a.dc = make_divconst(g);
    a.t = t;
    a.f = f;
    a.p = p;
    a.q = q;
    a.sp = sp;
    a.dep_cap = dep_cap;
    a.st = st;
    a.d = diff ? *diff : DiffArgs{};
    a.snap_on = diff && diff->snap.p[0] != nullptr;
    /* dynamic LDS: one 4-byte entry per line group */
    const size_t lds = (size_t)4 * t.TX * t.TY * t.TZ * ((p.cap + GS64 - 1) / GS64);
    const int nt = push_threads(t.ntiles);
    if (!diff && t.TZ == TZS) {
        if (t.ntiles <= 512)   /* two a CU: 51.1 against 52.0 us a step at 128 */
            hipLaunchKernelGGL((k_push_deposit<TXS, TYS, TZS, false, false, 512>),
                               dim3((unsigned)t.ntiles), dim3(512), lds, s, a);
        else                   /* 73.3 against 83.8 us at 1020 */
            hipLaunchKernelGGL((k_push_deposit<TXS, TYS, TZS, false, false, PIC_BLOCK>),
                               dim3((unsigned)t.ntiles), dim3(PIC_BLOCK), lds, s, a);
        return;
    }
    const bool tape = diff && diff->tape_mode != PIC_TAPE_OFF;
    auto launch = [&](auto diff_on, auto tape_on, auto threads) {
        constexpr int NT = decltype(threads)::value;
        hipLaunchKernelGGL((k_push_deposit<TXC, TYC, TZC, decltype(diff_on)::value,
                                           decltype(tape_on)::value, NT>),
                           dim3((unsigned)t.ntiles), dim3(NT), lds, s, a);
    };
    auto with_threads = [&](auto diff_on, auto tape_on) {
        if (nt == 1024) launch(diff_on, tape_on, std::integral_constant<int, 1024>());
        else if (nt == 512) launch(diff_on, tape_on, std::integral_constant<int, 512>());
        else launch(diff_on, tape_on, std::integral_constant<int, PIC_BLOCK>());
    };
    if (tape) with_threads(std::true_type(), std::true_type());
    else if (diff) with_threads(std::true_type(), std::false_type());
    else with_threads(std::false_type(), std::false_type());
}

void launch_jfix_to_f64(const Grid &g, FieldPtrs f, DiffArgs d, hipStream_t s) {
    hipLaunchKernelGGL(k_jfix_to_f64, dim3(blocks_for(g.G)), dim3(PIC_BLOCK), 0, s, g.G, f, d);
}

void launch_arrive_fold_f64(const Grid &g, const TileGeom &t, PartPtrs p, QueuePtrs q,
                            DevStatus *st, FieldPtrs f, long long *const jfix[3], int what,
                            hipStream_t s) {
    const unsigned tiles = what & PIC_ARRIVE ? (unsigned)t.ntiles : 0;
    const unsigned fold_end = tiles + (what & PIC_FOLD ? fold_blocks(g) : 0);
    const unsigned blocks = fold_end + (jfix ? blocks_for(g.G) : 0);
    FoldJ<double> J{};
    for (int k = 0; k < 3; k++) {
        J.J[k] = f.f[PIC_JX + k];
        if (jfix) J.fix[k] = jfix[k];
    }
    if (t.TZ == TZS)
        hipLaunchKernelGGL((k_arrive_fold<TXS, TYS, TZS, double>), dim3(blocks), dim3(PIC_BLOCK),
                           0, s, g, t, p, q, st, J, tiles, fold_end);
    else
        hipLaunchKernelGGL((k_arrive_fold<TXC, TYC, TZC, double>), dim3(blocks), dim3(PIC_BLOCK),
                           0, s, g, t, p, q, st, J, tiles, fold_end);
}

void launch_scatter_load(const long *offsets, long ncell, const double *src[6],
                         const unsigned char *srcsp, PartPtrs p, hipStream_t s) {
    hipLaunchKernelGGL(k_scatter_load, dim3(cell_blocks(ncell)), dim3(PIC_BLOCK), 0, s,
                       offsets, ncell, src[0], src[1], src[2], src[3], src[4], src[5], srcsp, p);
}

void launch_repack(long ncell, PartPtrs from, PartPtrs to, hipStream_t s) {
    hipLaunchKernelGGL(k_repack, dim3(blocks_for(ncell * from.cap)), dim3(PIC_BLOCK), 0, s, ncell,
                       from, to);
}

void launch_fix_arrivals(const TileGeom &t, QueuePtrs q, int oldcap, PartPtrs to, hipStream_t s) {
    hipLaunchKernelGGL(k_fix_arrivals, dim3((unsigned)t.ntiles), dim3(PIC_BLOCK), 0, s, q, oldcap,
                       to);
}

void launch_gather_particles(long ncell, const long *offsets, PartPtrs p, double *dst[6],
                             unsigned char *dsp, int *dcell, int *did, hipStream_t s) {
    hipLaunchKernelGGL(k_gather_particles, dim3(cell_blocks(ncell)), dim3(PIC_BLOCK), 0, s,
                       ncell, offsets, p, dst[0], dst[1], dst[2], dst[3], dst[4], dst[5], dsp,
                       dcell, did);
}

void launch_scatter_ids(const long *offsets, long ncell, const int *src, PartPtrs p,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_scatter_ids, dim3(cell_blocks(ncell)), dim3(PIC_BLOCK), 0, s,
                       offsets, ncell, src, p);
}

/* With few tiles the push lasts as long as the fullest CU takes: tiles of 16
 * cells spread a small box over more CUs and leave a shorter last round, for a
 * sixth more work per cell (halo nodes staged and flushed, workgroup starts).
 * So they are taken where 16 cells x rounds x 1.2 is below the large tiles' 64
 * cells x rounds, up to two large tiles a CU.  Whole steps, FP64, 32 to 51
 * particles per cell, us with large / small tiles:
 *   large tiles  32  66.6 / 51.1      256  64.4 / 64.5      483  96.8 /  99.0
 *                64  68.4 / 53.2      306  92.4 / 73.3      512  99.7 / 107.5
 *               128  61.4 / 54.2 */
TileGeom make_tile_geom(int Nx, int Ny, int Nz, bool small_ok) {
    auto tiles = [&](int X, int Y, int Z) {
        TileGeom t;
        t.TX = X;
        t.TY = Y;
        t.TZ = Z;
        t.ntx = (Nx + X - 1) / X;
        t.nty = (Ny + Y - 1) / Y;
        t.ntz = (Nz + Z - 1) / Z;
        t.ntiles = (long)t.ntx * t.nty * t.ntz;
        t.order = nullptr;
        return t;
    };
    constexpr long CUS = 256;
    auto cells_per_cu = [&](const TileGeom &t) {
        return (t.ntiles + CUS - 1) / CUS * t.TX * t.TY * t.TZ;
    };
    const TileGeom large = tiles(TXC, TYC, TZC), small = tiles(TXS, TYS, TZS);
    return small_ok && large.ntiles <= 2 * CUS && 6 * cells_per_cu(small) < 5 * cells_per_cu(large)
               ? small
               : large;
}
