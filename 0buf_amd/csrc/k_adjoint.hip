/*
 * k_adjoint.hip -- adjoint kernels of the FP64 step (differentiable form).
 *
 * Forward step t (s_{t-1} -> s_t, Plasma::Step, gpu_plasma.h:605-620):
 *     Q   = Ch E                     (MagneticStageOne, on the Q ranges)
 *     H'  = H + Q                    gather reads E and H'
 *     p1  = Boris(p, E(x), H'(x)),   x1 = x + tau u(p1)
 *     J   = VB deposit of x -> x1    (per segment pqr)
 *     x   = Reflect(x1)              (a shift: derivative 1)
 *     Jf  = Fold(J)
 *     H'' = H' + Q                   (same Q)
 *     E'  = P(E + Ce H'' - tau Jf)   (E ranges, then the periodic ghost copies)
 *     W_t = sum E'^2
 * The reverse step takes (lamE, lamH, lamP) at s_t to s_{t-1}:
 *   1. lamE += 2 w_t E_t                                (k_adj_seed_energy)
 *   2. lamE <- P^T lamE                                 (k_adj_e_periodic)
 *   3. lamH += Ce^T lamE|R ; lamQ := lamH|RQ ;
 *      lamJ := -tau lamE|R                              (k_adj_curl_e)
 *   4. lamJ <- Fold^T lamJ                              (k_adj_fold_j)
 *   5. particle adjoint: reverse deposit (a gather of lamJ), reverse push,
 *      reverse Boris, reverse gather (an atomic scatter into lamE, lamH)
 *                                                       (k_adj_particles)
 *   6. lamE += Ch^T (lamQ + lamH|RQ)                    (k_adj_curl_h)
 * after which lamH is the adjoint of H_{t-1} and lamE that of E_{t-1}.
 * Field transposes are gathers (one node per lane, deterministic); the
 * particle stage accumulates lamE, lamH in an LDS box per tile with FP64
 * atomics and adds the box to the global arrays with FP64 atomics.
 */
#include "k_fold.h"
#include "k_push_math.h"

#pragma clang fp contract(off)

namespace {

constexpr int TXC = 2, TYC = 4, TZC = 8;

/* Copies of the LDS adjoint box the gather adjoint scatters into, lane l
 * adding into copy l % ACOPIES, copies 9 mod 16 doubles apart (the reasons
 * stand at the FP32 adjoint's).  Measured, one step at 24.6M particles,
 * 128x64x64 cells, before the changes below: 2.54 ms with 5 copies, 2.61 with
 * 4, 2.83 with 3; 3.71 with 3 copies on the same banks.  6 copies of whole
 * boxes leave one workgroup per CU (86 KB). */
constexpr int ACOPIES = 5;
constexpr int copy_stride(int n) { return (n + 6) / 16 * 16 + 9; }   /* >= n, 9 mod 16 */

inline unsigned blocks_for(long n) { return (unsigned)((n + PIC_BLOCK - 1) / PIC_BLOCK); }

/* 32-bit arithmetic: the grid has fewer than 2^31 nodes */
__device__ __forceinline__ void decode32(const Grid &g, unsigned n, int &i, int &l, int &k) {
    const unsigned sy = (unsigned)g.sy, ny2 = (unsigned)(g.Ny + 2), t = n / sy;
    k = (int)(n - t * sy);
    const unsigned ii = t / ny2;
    l = (int)(t - ii * ny2);
    i = (int)ii;
}

__global__ __launch_bounds__(PIC_BLOCK) void k_adj_seed_energy(Grid g, const double *Ex,
                                                               const double *Ey, const double *Ez,
                                                               double w2, AdjLam l) {
    const long n = (long)blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (n >= g.G) return;
    l.E[0][n] += w2 * Ex[n];
    l.E[1][n] += w2 * Ey[n];
    l.E[2][n] += w2 * Ez[n];
}

/* transposes of the periodic E ghost copies, the forward's x, z and (in
 * ghost_mode 1) y copies last to first, E[0] = E[N]; E[N+1] = E[1] along a line
 * becoming L[N] += L[0], L[0] = 0; L[1] += L[N+1], L[N+1] = 0.  One thread per
 * class of nodes the copies combine (k_fold.h), one launch: three of their
 * own took 15 us of a small step.
 *   z: Ex over i in [0,Nx], l in [0,Ny+1]; Ey over i in [0,Nx+1], l in [0,Ny]
 *   x: Ey over l in [0,Ny], k in [1,Nz]; Ez over l in [1,Ny], k in [0,Nz]
 *   y (ghost_mode 1): Ex and Ez */
__global__ __launch_bounds__(PIC_BLOCK) void k_adj_e_periodic(Grid g, AdjLam lam) {
    const unsigned t = blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (t >= shell_count(g)) return;
    const NodeClass c = node_class(g, t);
    on_class(c, lam.E, [&](int cc, double (&v)[8]) {
        auto back = [&](int d, auto in_range) {
            class_pairs(c, v, d, [&](double &r, double &p, int s) {
                if (!in_range(s)) return;
                r += p;
                p = 0.0;
            });
        };
        if (g.ghost_mode == 1 && cc != 1) back(1, [](int) { return true; });
        if (cc == 0) back(2, [&](int s) { return c.i(s) <= g.Nx; });
        if (cc == 1) back(2, [&](int s) { return c.l(s) <= g.Ny; });
        if (cc == 1)
            back(0, [&](int s) { return c.l(s) <= g.Ny && c.k(s) >= 1 && c.k(s) <= g.Nz; });
        if (cc == 2)
            back(0, [&](int s) { return c.l(s) >= 1 && c.l(s) <= g.Ny && c.k(s) <= g.Nz; });
    });
}

/* E-update ranges (emeElement, kernels.cu:1162-1181) */
__device__ __forceinline__ bool in_ex(const Grid &g, int i, int l, int k) {
    return i >= 0 && i <= g.Nx && l >= 1 && l <= g.Ny && k >= 1 && k <= g.Nz;
}
__device__ __forceinline__ bool in_ey(const Grid &g, int i, int l, int k) {
    return i >= 1 && i <= g.Nx && l >= 0 && l <= g.Ny && k >= 1 && k <= g.Nz;
}
__device__ __forceinline__ bool in_ez(const Grid &g, int i, int l, int k) {
    return i >= 1 && i <= g.Nx && l >= 1 && l <= g.Ny && k >= 0 && k <= g.Nz;
}
/* Q ranges (emh1_Element, kernels.cu:1052-1089) */
__device__ __forceinline__ bool in_qx(const Grid &g, int i, int l, int k) {
    return i >= 0 && i <= g.Nx + 1 && l >= 0 && l <= g.Ny && k >= 0 && k <= g.Nz;
}
__device__ __forceinline__ bool in_qy(const Grid &g, int i, int l, int k) {
    return i >= 0 && i <= g.Nx && l >= 0 && l <= g.Ny + 1 && k >= 0 && k <= g.Nz;
}
__device__ __forceinline__ bool in_qz(const Grid &g, int i, int l, int k) {
    return i >= 0 && i <= g.Nx && l >= 0 && l <= g.Ny && k >= 0 && k <= g.Nz + 1;
}

/* transpose of the E update  E += c1y(Hz - Hz[l-1]) - c1z(Hy - Hy[k-1]) - tau Jx  etc.
 * per H node; also lamJ = -tau lamE on the E ranges and lamQ = lamH'' on the
 * Q ranges */
__global__ __launch_bounds__(PIC_BLOCK) void k_adj_curl_e(Grid g, AdjLam lam) {
    const long n = (long)blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (n >= g.G) return;
    int i, l, k;
    decode32(g, (unsigned)n, i, l, k);
    const double c1x = g.tau / g.hx, c1y = g.tau / g.hy, c1z = g.tau / g.hz, tau = g.tau;
    const double *LEx = lam.E[0], *LEy = lam.E[1], *LEz = lam.E[2];
    const long sy = g.sy, sx = g.sx;
    /* every load first (the node itself past the end), then the ranges: behind
     * the tests they were waited for in turn */
    const long nl = n + sy < g.G ? n + sy : n, nk = n + 1 < g.G ? n + 1 : n,
               ni = n + sx < g.G ? n + sx : n;
    const double vx = LEx[n], vy = LEy[n], vz = LEz[n], vxl = LEx[nl], vxk = LEx[nk],
                 vyi = LEy[ni], vyk = LEy[nk], vzi = LEz[ni], vzl = LEz[nl];
    const double H0 = lam.H[0][n], H1 = lam.H[1][n], H2 = lam.H[2][n];
    const double ex = in_ex(g, i, l, k) ? vx : 0.0;
    const double ey = in_ey(g, i, l, k) ? vy : 0.0;
    const double ez = in_ez(g, i, l, k) ? vz : 0.0;
    const double ex_l = in_ex(g, i, l + 1, k) ? vxl : 0.0;
    const double ex_k = in_ex(g, i, l, k + 1) ? vxk : 0.0;
    const double ey_i = in_ey(g, i + 1, l, k) ? vyi : 0.0;
    const double ey_k = in_ey(g, i, l, k + 1) ? vyk : 0.0;
    const double ez_i = in_ez(g, i + 1, l, k) ? vzi : 0.0;
    const double ez_l = in_ez(g, i, l + 1, k) ? vzl : 0.0;
    const double hx = H0 + (c1z * (ey - ey_k) - c1y * (ez - ez_l));
    const double hy = H1 + (-c1z * (ex - ex_k) + c1x * (ez - ez_i));
    const double hz = H2 + (c1y * (ex - ex_l) - c1x * (ey - ey_i));
    lam.H[0][n] = hx;
    lam.H[1][n] = hy;
    lam.H[2][n] = hz;
    lam.Q[0][n] = in_qx(g, i, l, k) ? hx : 0.0;
    lam.Q[1][n] = in_qy(g, i, l, k) ? hy : 0.0;
    lam.Q[2][n] = in_qz(g, i, l, k) ? hz : 0.0;
    lam.J[0][n] = -tau * ex;
    lam.J[1][n] = -tau * ey;
    lam.J[2][n] = -tau * ez;
}

/* transpose of the J fold (k_fold_j, per axis and component: if axis != c:
 * J[1] += J[N+1]; if !(axis == y && c == y): J[N+1] = J[1]; J[0] += J[N];
 * J[N] = J[0]), operations reversed, z, y, x; one thread per class of nodes the
 * fold combines, one launch instead of three */
__global__ __launch_bounds__(PIC_BLOCK) void k_adj_fold_j(Grid g, AdjLam lam) {
    const unsigned t = blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (t >= shell_count(g)) return;
    const NodeClass c = node_class(g, t);
    const bool at_n[3] = {c.ri == g.Nx, c.rl == g.Ny, c.rk == g.Nz};
    on_class(c, lam.J, [&](int cc, double (&v)[8]) {
#pragma unroll
        for (int d = 2; d >= 0; d--)
            class_pairs(c, v, d, [&](double &r, double &p, int) {
                if (at_n[d] || d != cc) {          /* both ends take the sum */
                    r += p;
                    p = r;
                } else if (d != 1) {
                    r += p;
                    p = 0.0;
                }
            });
    });
}

/* transpose of Q = Ch E:  Qx = 1/2(c1z(Ey[k+1]-Ey) - c1y(Ez[l+1]-Ez)) etc.,
 * with the Q adjoint mu = lamQ + lamH on the Q ranges */
__global__ __launch_bounds__(PIC_BLOCK) void k_adj_curl_h(Grid g, AdjLam lam) {
    const long n = (long)blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (n >= g.G) return;
    int i, l, k;
    decode32(g, (unsigned)n, i, l, k);
    const double c1x = g.tau / g.hx, c1y = g.tau / g.hy, c1z = g.tau / g.hz;
    const long sy = g.sy, sx = g.sx;
    /* every load first (the node itself where a neighbour is missing) */
    const long nk = k >= 1 ? n - 1 : n, nl = l >= 1 ? n - sy : n, ni = i >= 1 ? n - sx : n;
    auto mu = [&](int d, long m) { return lam.Q[d][m] + lam.H[d][m]; };
    const double x = mu(0, n), y = mu(1, n), z = mu(2, n), xk = mu(0, nk), xl = mu(0, nl),
                 yk = mu(1, nk), yi = mu(1, ni), zl = mu(2, nl), zi = mu(2, ni);
    const double E0 = lam.E[0][n], E1 = lam.E[1][n], E2 = lam.E[2][n];
    const double mx = in_qx(g, i, l, k) ? x : 0.0, my = in_qy(g, i, l, k) ? y : 0.0,
                 mz = in_qz(g, i, l, k) ? z : 0.0;
    const double mx_k = k >= 1 && in_qx(g, i, l, k - 1) ? xk : 0.0;
    const double mx_l = l >= 1 && in_qx(g, i, l - 1, k) ? xl : 0.0;
    const double my_k = k >= 1 && in_qy(g, i, l, k - 1) ? yk : 0.0;
    const double my_i = i >= 1 && in_qy(g, i - 1, l, k) ? yi : 0.0;
    const double mz_l = l >= 1 && in_qz(g, i, l - 1, k) ? zl : 0.0;
    const double mz_i = i >= 1 && in_qz(g, i - 1, l, k) ? zi : 0.0;
    lam.E[0][n] = E0 + 0.5 * (c1z * (my - my_k) + c1y * (mz_l - mz));
    lam.E[1][n] = E1 + 0.5 * (c1z * (mx_k - mx) + c1x * (mz - mz_i));
    lam.E[2][n] = E2 + 0.5 * (c1y * (mx - mx_l) + c1x * (my_i - my));
}

/* ---------------------------------------------------------------- particles */

struct AdjArgs {
    Grid g;
    DivConst dc;
    TileGeom t;
    AdjFwd fwd;
    PartPtrs p;          /* compact record of s_{t-1} */
    const long *snap_off;
    SpeciesTable sp;
    AdjLam lam;
    LamParts lp;
    DevStatus *st;
};

/* adjoint of one pqr segment (cell.h:1511-1693): gradient of
 * sum_nodes lamJ[node] * contribution(A -> B) with respect to the segment
 * ends A and B; lamJ is read from the LDS box at the forward's nodes */
template <int BY, int BZ, int JY0, int JZ0>
__device__ __forceinline__ void pqr_adj(const double *sL, const Geo &c, const DivConst &dc, int ix,
                                        int iy, int iz, double ax, double ay, double az, double bx,
                                        double by, double bz, double q, double gA[3],
                                        double gB[3]) {
#pragma clang fp contract(fast)   /* no decision depends on the reverse sweep */
    const double dx = 0.50 * (ax + bx) - c.hx * ((double)ix - 2.50);
    const double dy = 0.50 * (ay + by) - c.hy * ((double)iy - 2.50);
    const double dz = 0.50 * (az + bz) - c.hz * ((double)iz - 2.50);
    const double dx1 = c.hx - dx, dy1 = c.hy - dy, dz1 = c.hz - dz;
    const double Dx = bx - ax, Dy = by - ay, Dz = bz - az;
    const double s1 = Dy * Dz * dc.r12, s2 = Dx * Dz * dc.r12, s3 = Dx * Dy * dc.r12;
    /* the forward deposits nothing outside the tile stencil (and flags it):
     * weight 0, at a node inside the box.  (An early return would put gA and
     * gB in scratch memory.) */
    const bool in = (unsigned)((ix - 2) | (iy - 2) | (iz - 2)) <= 1u;
    const double qi = in ? q : 0.0;
    const double kx = qi * dc.rDx, ky = qi * dc.rDy, kz = qi * dc.rDz;
    const double SU = Dx * kx, SV = Dy * ky, SW = Dz * kz;
    const int n = in ? c.n0 + (ix != 2 ? BY * BZ : 0) + (iy != 2 ? BZ : 0) + iz - 2 : 0;
    const double *Lx = sL, *Ly = sL + JY0, *Lz = sL + JZ0;
    const double a0 = Lx[n], a1 = Lx[n + 1], a2 = Lx[n + BZ], a3 = Lx[n + BZ + 1];
    const double b0 = Ly[n], b1 = Ly[n + 1], b2 = Ly[n + BY * BZ], b3 = Ly[n + BY * BZ + 1];
    const double c0 = Lz[n], c1 = Lz[n + BZ], c2 = Lz[n + BY * BZ], c3 = Lz[n + BY * BZ + BZ];
    const double Bx = a0 * (dy1 * dz1 + s1) + a1 * (dy1 * dz - s1) + a2 * (dy * dz1 - s1) +
                      a3 * (dy * dz + s1);
    const double By = b0 * (dx1 * dz1 + s2) + b1 * (dx1 * dz - s2) + b2 * (dx * dz1 - s2) +
                      b3 * (dx * dz + s2);
    const double Bz = c0 * (dx1 * dy1 + s3) + c1 * (dx1 * dy - s3) + c2 * (dx * dy1 - s3) +
                      c3 * (dx * dy + s3);
    const double Bx_dy = -a0 * dz1 - a1 * dz + a2 * dz1 + a3 * dz;
    const double Bx_dz = -a0 * dy1 + a1 * dy1 - a2 * dy + a3 * dy;
    const double Bx_s = a0 - a1 - a2 + a3;
    const double By_dx = -b0 * dz1 - b1 * dz + b2 * dz1 + b3 * dz;
    const double By_dz = -b0 * dx1 + b1 * dx1 - b2 * dx + b3 * dx;
    const double By_s = b0 - b1 - b2 + b3;
    const double Bz_dx = -c0 * dy1 - c1 * dy + c2 * dy1 + c3 * dy;
    const double Bz_dy = -c0 * dx1 + c1 * dx1 - c2 * dx + c3 * dx;
    const double Bz_s = c0 - c1 - c2 + c3;
    /* d/d(midpoint offsets) and d/d(segment deltas) */
    const double gdx = SV * By_dx + SW * Bz_dx;
    const double gdy = SU * Bx_dy + SW * Bz_dy;
    const double gdz = SU * Bx_dz + SV * By_dz;
    const double gDx = kx * Bx + (SV * By_s * Dz + SW * Bz_s * Dy) * dc.r12;
    const double gDy = ky * By + (SU * Bx_s * Dz + SW * Bz_s * Dx) * dc.r12;
    const double gDz = kz * Bz + (SU * Bx_s * Dy + SV * By_s * Dx) * dc.r12;
    gA[0] = 0.5 * gdx - gDx;
    gA[1] = 0.5 * gdy - gDy;
    gA[2] = 0.5 * gdz - gDz;
    gB[0] = 0.5 * gdx + gDx;
    gB[1] = 0.5 * gdy + gDy;
    gB[2] = 0.5 * gdz + gDz;
}

/* Interpolate3D with the forward's rounding sequence (interp, k_push_math.h),
 * and the derivatives of the value with respect to the far-plane weights sx1,
 * sy1, sz1 (the near ones are 1 minus them), from the same eight nodes: the
 * reverse part needs no node again */
template <int BY, int BZ>
__device__ __forceinline__ double interp_grad(const double *F, int o, double sx1, double sy1,
                                              double sz1, double g[3]) {
    const double f00 = F[o], f01 = F[o + BZ], f10 = F[o + BY * BZ], f11 = F[o + BY * BZ + BZ];
    const double d00 = F[o + 1] - f00, d01 = F[o + BZ + 1] - f01;
    const double d10 = F[o + BY * BZ + 1] - f10, d11 = F[o + BY * BZ + BZ + 1] - f11;
    const double z00 = fma(sz1, d00, f00), z01 = fma(sz1, d01, f01);
    const double z10 = fma(sz1, d10, f10), z11 = fma(sz1, d11, f11);
    const double e0 = z01 - z00, e1 = z11 - z10;
    const double y0 = fma(sy1, e0, z00), y1 = fma(sy1, e1, z10);
    const double dy0 = fma(sy1, d01 - d00, d00), dy1 = fma(sy1, d11 - d10, d10);
    g[0] = y1 - y0;
    g[1] = fma(sx1, e1 - e0, e0);
    g[2] = fma(sx1, dy1 - dy0, dy0);
    return fma(sx1, g[0], y0);
}

/* its adjoint: lam * weight into the eight nodes of the LDS adjoint box */
template <int BY, int BZ>
__device__ __forceinline__ void interp_scatter(double *A, int o, double sx, double sx1, double sy,
                                               double sy1, double sz, double sz1, double lam) {
    const double yz00 = sy * sz, yz01 = sy * sz1, yz10 = sy1 * sz, yz11 = sy1 * sz1;
    const double lx0 = lam * sx, lx1 = lam * sx1;
    atomicAdd(&A[o], lx0 * yz00);
    atomicAdd(&A[o + 1], lx0 * yz01);
    atomicAdd(&A[o + BZ], lx0 * yz10);
    atomicAdd(&A[o + BZ + 1], lx0 * yz11);
    atomicAdd(&A[o + BY * BZ], lx1 * yz00);
    atomicAdd(&A[o + BY * BZ + 1], lx1 * yz01);
    atomicAdd(&A[o + BY * BZ + BZ], lx1 * yz10);
    atomicAdd(&A[o + BY * BZ + BZ + 1], lx1 * yz11);
}

__device__ __forceinline__ void cross(const double a[3], const double b[3], double r[3]) {
#pragma clang fp contract(fast)
    r[0] = a[1] * b[2] - a[2] * b[1];
    r[1] = a[2] * b[0] - a[0] * b[2];
    r[2] = a[0] * b[1] - a[1] * b[0];
}
__device__ __forceinline__ double dot3(const double a[3], const double b[3]) {
#pragma clang fp contract(fast)
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

template <int TX, int TY, int TZ, int NT>
__global__ __launch_bounds__(NT) void k_adj_particles(AdjArgs a) {
    constexpr int C = TX * TY * TZ;
    constexpr int BX = TX + 2, BY = TY + 2, BZ = TZ + 2, NB = BX * BY * BZ;
    /* Every field component takes all BX planes: a particle exactly on its
     * cell's upper face stays in the cell (flyDirection's v > v0 + h), and its
     * node-type components then read the planes behind that face, TX and TX + 1
     * in the tile's last cell.  (FP32 offsets stay below 1; their boxes end
     * earlier.)  Jx, dual along x, is read at planes 0..TX only. */
    constexpr int NBX = (TX + 1) * BY * BZ;
    constexpr int NF = 6 * NB, NJ = NBX + 2 * NB, JY0 = NBX, JZ0 = NBX + NB;
    constexpr int LB[3] = {0, JY0, JZ0}, LN[3] = {NBX, NB, NB};   /* lamJ: start, nodes */
    constexpr int AS = copy_stride(NF);
    static_assert(AS >= NF && AS % 16 == 9, "");
    __shared__ double sF[NF];        /* E, H' of the forward step */
    __shared__ double sL[NJ];        /* lamJ */
    __shared__ double sA[ACOPIES * AS];   /* lamE, lamH' accumulated by the gather adjoint */
    double *const myA = sA + (threadIdx.x % ACOPIES) * AS;
    __shared__ int sOff[C + 1];
    __shared__ int sCnt[C];
    __shared__ unsigned sFlags;

    const Grid &g = a.g;
    const int tid = threadIdx.x;
    const TileAt at = tile_of_block(a.t, blockIdx.x);
    const long tile = at.tile;
    const int tx = at.tx, ty = at.ty, tz = at.tz;
    const int I0 = tx * TX, L0 = ty * TY, K0 = tz * TZ;
    const int cap = a.p.cap;

    /* thread n takes box node n of every box (one decode, one 32-bit
     * offset: the grid has fewer than 2^31 nodes) and cell n of the tile;
     * every global load is issued before the first LDS write */
    static_assert(NB <= NT && C <= NT, "one box node and one cell per thread");
    const double *const Fsrc[6] = {a.fwd.E[0], a.fwd.E[1], a.fwd.E[2],
                                   a.fwd.H[0], a.fwd.H[1], a.fwd.H[2]};
    const int nu = tid / (BY * BZ), nv = (tid / BZ) % BY, nw = tid % BZ;
    const bool node_in = tid < NB && I0 + nu <= g.Nx + 1 && L0 + nv <= g.Ny + 1 &&
                         K0 + nw <= g.Nz + 1;
    const unsigned noff = (unsigned)(I0 + nu) * g.sx + (unsigned)(L0 + nv) * g.sy + (K0 + nw);
    {
        double fv[6], lj[3];
#pragma unroll
        for (int q = 0; q < 6; q++) fv[q] = 0.0;
#pragma unroll
        for (int q = 0; q < 3; q++) lj[q] = 0.0;
        if (node_in) {
#pragma unroll
            for (int q = 0; q < 6; q++) fv[q] = Fsrc[q][noff];
#pragma unroll
            for (int q = 0; q < 3; q++) lj[q] = a.lam.J[q][noff];
        }
        const int gi = I0 + tid / (TY * TZ), gl = L0 + (tid / TZ) % TY, gk = K0 + tid % TZ;
        int cnt = 0;
        if (tid < C && gi < g.Nx && gl < g.Ny && gk < g.Nz) {
            cnt = a.p.count[((long)gi * g.Ny + gl) * g.Nz + gk];
            cnt = cnt < cap ? cnt : cap;
        }
        if (tid < NB) {
#pragma unroll
            for (int q = 0; q < 6; q++) sF[q * NB + tid] = fv[q];
#pragma unroll
            for (int q = 0; q < 3; q++)
                if (tid < LN[q]) sL[LB[q] + tid] = lj[q];
        }
        if (tid < C) sCnt[tid] = cnt;
    }
    for (int e = tid; e < ACOPIES * AS; e += NT) sA[e] = 0.0;
    if (tid == 0) sFlags = 0;
    __syncthreads();
    static_assert(C == 64, "one wavefront scans the tile's cells");
    if (tid < 64) {
        int total;
        sOff[tid] = wave_excl_scan(sCnt[tid], total);
        if (tid == 0) sOff[C] = total;
    }
    __syncthreads();
    const int T = sOff[C];
    const long rec0 = uniform(a.snap_off[tile]);

    const double hx = g.hx, hy = g.hy, hz = g.hz, tau = g.tau;
    unsigned bad = 0;
    for (int fidx = tid; fidx < T; fidx += NT) {
        int lo = 0, hi = C;
        while (hi - lo > 1) {
            int mid = (lo + hi) >> 1;
            if (sOff[mid] <= fidx) lo = mid; else hi = mid;
        }
        const int c = lo;
        const int ca = c / (TY * TZ), cb = (c / TZ) % TY, cc = c % TZ;
        const int gi = I0 + ca, gl = L0 + cb, gk = K0 + cc;
        const long pidx = rec0 + fidx;    /* compact record */
        Geo G;
        G.n0 = (ca * BY + cb) * BZ + cc;
        G.hx = hx; G.hy = hy; G.hz = hz;
        const double x0 = (double)gi * hx, y0 = (double)gl * hy, z0 = (double)gk * hz;

        const double x = a.p.p[0][pidx], y = a.p.p[1][pidx], z = a.p.p[2][pidx];
        const double pu = a.p.p[3][pidx], pv = a.p.p[4][pidx], pw = a.p.p[5][pidx];
        const unsigned char s = a.p.sp[pidx];
        const int pid = a.p.id[pidx];
        const double mass = a.sp.m[s], q_m = a.sp.q_m[s];
        const double tau1 = q_m * tau * 0.5;

        /* ---- forward recompute, the push kernel's arithmetic ---- */
        const double xl = x - x0, yl = y - y0, zl = z - z0;
        const double frx = divc(xl, hx, a.dc.rhx);
        const double fry = divc(yl, hy, a.dc.rhy);
        const double frz = divc(zl, hz, a.dc.rhz);
        double Ef[3] = {0, 0, 0}, Hf[3] = {0, 0, 0};
        int o[6] = {0, 0, 0, 0, 0, 0};
        double gw[6][3] = {};   /* d(field component) / d(far weights) */
        const bool live = !(x < 0 || y < 0 || z < 0);
        GatherIdx W{};
        if (live) {
            W = gather_index(x, y, z, frx, fry, frz, g, a.dc);
            if (!W.ok) {
                bad = 1;
            } else {
                const double s11 = 1. - W.s1, s21 = 1. - W.s2, s31 = 1. - W.s3, s41 = 1. - W.s4,
                             s51 = 1. - W.s5, s61 = 1. - W.s6;
                /* node of the component's near corner in its box */
                const int X = G.n0 + (W.ix != 2 ? BY * BZ : 0),
                          X1 = G.n0 + (W.i1x != 2 ? BY * BZ : 0),
                          Y = W.iy != 2 ? BZ : 0, Y1 = W.i1y != 2 ? BZ : 0, Z = W.iz - 2,
                          Z1 = W.i1z - 2;
                o[0] = X + Y1 + Z1;
                Ef[0] = interp_grad<BY, BZ>(sF + 0 * NB, o[0], s11, s41, s61, gw[0]);
                o[1] = X1 + Y + Z1;
                Ef[1] = interp_grad<BY, BZ>(sF + 1 * NB, o[1], s21, s31, s61, gw[1]);
                o[2] = X1 + Y1 + Z;
                Ef[2] = interp_grad<BY, BZ>(sF + 2 * NB, o[2], s21, s41, s51, gw[2]);
                o[3] = X1 + Y + Z;
                Hf[0] = interp_grad<BY, BZ>(sF + 3 * NB, o[3], s21, s31, s51, gw[3]);
                o[4] = X + Y1 + Z;
                Hf[1] = interp_grad<BY, BZ>(sF + 4 * NB, o[4], s11, s41, s51, gw[4]);
                o[5] = X + Y + Z1;
                Hf[2] = interp_grad<BY, BZ>(sF + 5 * NB, o[5], s11, s31, s61, gw[5]);
            }
        }
        const Boris B = boris_move<true>(pu, pv, pw, Ef[0], Ef[1], Ef[2], Hf[0], Hf[1], Hf[2], tau1);
        const double x1 = advance<true>(x, tau, B.g2, B.p1[0]) - x0,
                     y1 = advance<true>(y, tau, B.g2, B.p1[1]) - y0,
                     z1 = advance<true>(z, tau, B.g2, B.p1[2]) - z0;
        const Relay R = relay_point(xl, yl, zl, x1, y1, z1, frx, fry, frz,
                                    divc(x1, hx, a.dc.rhx), divc(y1, hy, a.dc.rhy),
                                    divc(z1, hz, a.dc.rhz), G);
        const int m = R.m;

        /* ---- reverse (contracted: no decision depends on it) ---- */
        double2 *const lq = (double2 *)(a.lp.v + (long)pid * PIC_LSTRIDE);
        const double2 q0 = lq[0], q1 = lq[1], q2 = lq[2];
        double lx1[3] = {q0.x, q0.y, q1.x};
        double lp1[3] = {q1.y, q2.x, q2.y};
        double lx[3];
        const double X0[3] = {xl, yl, zl}, X1[3] = {x1, y1, z1};
        /* deposit: J = pqr(i1; x -> e1) + [m != 0] pqr(i2; x2 -> x1) */
        {
#pragma clang fp contract(fast)
            double gA[3], gB[3];
            const double e1x = m ? R.x2x : x1, e1y = m ? R.x2y : y1, e1z = m ? R.x2z : z1;
            pqr_adj<BY, BZ, JY0, JZ0>(sL, G, a.dc, R.i1x, R.i1y, R.i1z, xl, yl, zl, e1x, e1y, e1z, mass,
                                gA, gB);
            lx[0] = gA[0];
            lx[1] = gA[1];
            lx[2] = gA[2];
            if (m == 0) {
                lx1[0] += gB[0];
                lx1[1] += gB[1];
                lx1[2] += gB[2];
            } else {
                double hA[3], hB[3];
                pqr_adj<BY, BZ, JY0, JZ0>(sL, G, a.dc, R.i2x, R.i2y, R.i2z, R.x2x, R.x2y, R.x2z, x1, y1,
                                    z1, mass, hA, hB);
                lx1[0] += hB[0];
                lx1[1] += hB[1];
                lx1[2] += hB[2];
                /* relay point x2(x, x1): crossed axes sit on a face (constant),
                 * the others on the straight path at sr = num/den */
                const double lx2[3] = {gB[0] + hA[0], gB[1] + hA[1], gB[2] + hA[2]};
                const bool cr[3] = {(m & 4) != 0, (m & 2) != 0, (m & 1) != 0};
                const double F[3] = {R.fx, R.fy, R.fz};
                double lsr = 0.0;
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const double v = cr[d] ? 0.0 : lx2[d];
                    lsr += v * (X1[d] - X0[d]);
                    lx[d] += v * (1.0 - R.sr);
                    lx1[d] += v * R.sr;
                }
                /* sr = num/den over the one or two crossed faces, num = sum
                 * (f_d - x_d) D_d, den = sum D_d^2.  (Selected, not branched
                 * around: a branch per axis became a computed index, which
                 * put the arrays in scratch memory.) */
                const double w = m != 7 ? lsr / R.den : 0.0;
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const double D = X1[d] - X0[d], f = F[d] - X0[d];
                    const double gx = 2.0 * R.sr * D - D - f, gx1 = f - 2.0 * R.sr * D;
                    lx[d] += cr[d] ? w * gx : 0.0;
                    lx1[d] += cr[d] ? w * gx1 : 0.0;
                }
            }
        }
        /* x1 = x + tau g2 p1 */
        for (int d = 0; d < 3; d++) lx[d] += lx1[d];
        {
#pragma clang fp contract(fast)
            const double lu[3] = {tau * lx1[0], tau * lx1[1], tau * lx1[2]};
            const double g2 = B.g2, g23 = g2 * g2 * g2;
            const double pl = dot3(B.p1, lu);
            for (int d = 0; d < 3; d++) lp1[d] += g2 * lu[d] - g23 * pl * B.p1[d];
        }
        /* p1 = pp + tau1 E;  pp = (s + (b.s) b + s x b) / (1 + b.b) */
        double lE[3], lH[3], lpm[3];
        {
#pragma clang fp contract(fast)
            for (int d = 0; d < 3; d++) lE[d] = tau1 * lp1[d];
            const double *b = B.b, *sv = B.s;
            const double rD = 1.0 / B.sden;
            double lN[3] = {lp1[0] * rD, lp1[1] * rD, lp1[2] * rD};
            /* pp recomputed from s and b for the denominator term */
            double sxb[3];
            cross(sv, b, sxb);
            const double bs = dot3(b, sv);
            double pp[3];
            for (int d = 0; d < 3; d++) pp[d] = (sv[d] + bs * b[d] + sxb[d]) * rD;
            const double bl = dot3(b, lN), lpp = dot3(lp1, pp);
            double bxl[3], lxs[3];
            cross(b, lN, bxl);
            cross(lN, sv, lxs);
            double ls[3], lb[3];
            for (int d = 0; d < 3; d++) {
                ls[d] = lN[d] + b[d] * bl + bxl[d];
                lb[d] = sv[d] * bl + bs * lN[d] + lxs[d] - 2.0 * lpp * rD * b[d];
            }
            /* s = pm + pm x b */
            double bxls[3], lsxpm[3];
            cross(b, ls, bxls);
            cross(ls, B.pm, lsxpm);
            for (int d = 0; d < 3; d++) {
                lpm[d] = ls[d] + bxls[d];
                lb[d] += lsxpm[d];
            }
            /* b = ps H, ps = tau1 g1, g1 = (pm.pm + 1)^-1/2 */
            const double lps = dot3(lb, Hf);
            for (int d = 0; d < 3; d++) lH[d] = B.ps * lb[d];
            if (tau1 != 0.0) {
                const double g1 = B.ps / tau1;
                const double k = -tau1 * g1 * g1 * g1 * lps;
                for (int d = 0; d < 3; d++) lpm[d] += k * B.pm[d];
            }
            /* pm = p + tau1 E */
            for (int d = 0; d < 3; d++) lE[d] += tau1 * lpm[d];
        }
        /* gather: scatter into the adjoint box, position derivative through
         * the weights (every far weight has d/dx = 1/h) */
        if (live && W.ok) {
            interp_scatter<BY, BZ>(myA + 0 * NB, o[0], W.s1, 1. - W.s1, W.s4, 1. - W.s4, W.s6,
                                   1. - W.s6, lE[0]);
            interp_scatter<BY, BZ>(myA + 1 * NB, o[1], W.s2, 1. - W.s2, W.s3, 1. - W.s3, W.s6,
                                   1. - W.s6, lE[1]);
            interp_scatter<BY, BZ>(myA + 2 * NB, o[2], W.s2, 1. - W.s2, W.s4, 1. - W.s4, W.s5,
                                   1. - W.s5, lE[2]);
            interp_scatter<BY, BZ>(myA + 3 * NB, o[3], W.s2, 1. - W.s2, W.s3, 1. - W.s3, W.s5,
                                   1. - W.s5, lH[0]);
            interp_scatter<BY, BZ>(myA + 4 * NB, o[4], W.s1, 1. - W.s1, W.s4, 1. - W.s4, W.s5,
                                   1. - W.s5, lH[1]);
            interp_scatter<BY, BZ>(myA + 5 * NB, o[5], W.s1, 1. - W.s1, W.s3, 1. - W.s3, W.s6,
                                   1. - W.s6, lH[2]);
            const double rh[3] = {a.dc.rhx, a.dc.rhy, a.dc.rhz};
            for (int d = 0; d < 3; d++) {
#pragma clang fp contract(fast)
                const double ds = lE[0] * gw[0][d] + lE[1] * gw[1][d] + lE[2] * gw[2][d] +
                                  lH[0] * gw[3][d] + lH[1] * gw[4][d] + lH[2] * gw[5][d];
                lx[d] += ds * rh[d];
            }
        }
        lq[0] = make_double2(lx[0], lx[1]);
        lq[1] = make_double2(lx[2], lpm[0]);
        lq[2] = make_double2(lpm[1], lpm[2]);
    }
    if (bad) atomicOr(&sFlags, (unsigned)PIC_F_RANGE);
    __syncthreads();
    if (tid < NB) {   /* thread n adds box node n of the six adjoint boxes */
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const int e = q * NB + tid;
            double val = sA[e];
            for (int r = 1; r < ACOPIES; r++) val += sA[r * AS + e];
            if (val != 0.0 && node_in)
                atomicAdd(q < 3 ? &a.lam.E[q][noff] : &a.lam.H[q - 3][noff], val);
        }
    }
    if (tid == 0 && sFlags) atomicOr(&a.st->flags, sFlags);
}

/* bitwise comparison of a recomputed array with its checkpoint */
template <typename T>
__global__ __launch_bounds__(PIC_BLOCK) void k_mismatch(const T *a, const T *b, long n,
                                                        DevStatus *st) {
    const long e = (long)blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (e < n && a[e] != b[e]) atomicOr(&st->flags, (unsigned)PIC_F_RECOMPUTE);
}

}  // namespace

void launch_mismatch(const void *a, const void *b, long n, int elem_bytes, DevStatus *st,
                     hipStream_t s) {
    if (elem_bytes == 8)
        hipLaunchKernelGGL(k_mismatch<unsigned long long>, dim3(blocks_for(n)), dim3(PIC_BLOCK),
                           0, s, (const unsigned long long *)a, (const unsigned long long *)b, n,
                           st);
    else
        hipLaunchKernelGGL(k_mismatch<unsigned int>, dim3(blocks_for(n)), dim3(PIC_BLOCK), 0, s,
                           (const unsigned int *)a, (const unsigned int *)b, n, st);
}

void launch_adj_seed_energy(const Grid &g, const double *const E[3], double w, AdjLam l,
                            hipStream_t s) {
    hipLaunchKernelGGL(k_adj_seed_energy, dim3(blocks_for(g.G)), dim3(PIC_BLOCK), 0, s, g, E[0],
                       E[1], E[2], 2.0 * w, l);
}

void launch_adj_e_periodic(const Grid &g, AdjLam l, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_e_periodic, dim3(fold_blocks(g)), dim3(PIC_BLOCK), 0, s, g, l);
}

void launch_adj_curl_e(const Grid &g, AdjLam l, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_curl_e, dim3(blocks_for(g.G)), dim3(PIC_BLOCK), 0, s, g, l);
}

void launch_adj_fold_j(const Grid &g, AdjLam l, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_fold_j, dim3(fold_blocks(g)), dim3(PIC_BLOCK), 0, s, g, l);
}

void launch_adj_particles_f64(const Grid &g, const TileGeom &t, AdjFwd fwd, PartPtrs snap,
                              const long *snap_off, SpeciesTable sp, AdjLam l, LamParts lp,
                              DevStatus *st, hipStream_t s) {
    AdjArgs a;
    a.g = g;
    a.dc = make_divconst(g);
    a.t = t;
    a.fwd = fwd;
    a.p = snap;
    a.snap_off = snap_off;
    a.sp = sp;
    a.lam = l;
    a.lp = lp;
    a.st = st;
    /* two wavefronts per SIMD at one tile per CU, as many as the registers
     * allow: 151 against 176 us at 256 tiles of 48 particles per cell; from two
     * tiles per CU on no gain (250 us either way at 512 tiles) */
    if (t.ntiles <= 256)
        hipLaunchKernelGGL((k_adj_particles<TXC, TYC, TZC, 512>), dim3((unsigned)t.ntiles), dim3(512), 0, s, a);
    else
        hipLaunchKernelGGL((k_adj_particles<TXC, TYC, TZC, PIC_BLOCK>), dim3((unsigned)t.ntiles),
                           dim3(PIC_BLOCK), 0, s, a);
}

void launch_adj_curl_h(const Grid &g, AdjLam l, hipStream_t s) {
    hipLaunchKernelGGL(k_adj_curl_h, dim3(blocks_for(g.G)), dim3(PIC_BLOCK), 0, s, g, l);
}
