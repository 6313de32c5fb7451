/*
 * k_push_math.h -- per-particle arithmetic of the FP64 step, shared by the
 * push kernel (k_particles_f64.hip) and the particle adjoint
 * (k_adjoint.hip).  The adjoint recomputes the forward step from a snapshot
 * with exactly these functions, so its gather indices, crossing code and
 * relay points are the forward's bit for bit.
 *
 * Both files are built with -ffp-contract=off and write the multiply-adds they
 * want fused as fma, so both kernels round alike.  In the plain form the new
 * momenta and positions keep the reference's rounding sequence (cell.h,
 * particle.h; its quotients and powers as divc and pow_m05 give them), as the
 * decisions (cells, weight floors, directions) do in both forms; the segment weights, and in the differentiable form the interpolation
 * and the rotation, are fused, with fewer roundings than the reference's.
 */
#ifndef K_PUSH_MATH_H
#define K_PUSH_MATH_H

#include "pic_internal.h"

/* Divisors that are constant over a run, with their correctly rounded
 * reciprocals: q = divc(x, d, r) returns the correctly rounded x/d in three
 * instructions (Markstein: q0 = x r, exact remainder x - q0 d by FMA, one
 * FMA correction), bit-identical to IEEE division.  From a reciprocal that is
 * only within an ulp (recip) the theorem's premise fails: the sum before the
 * last rounding is then within 2^-52 ulp of x/d, and the quotient is the
 * correctly rounded one unless x/d lies that close to a tie (none of 10^8
 * random quotients, nor of 10^8 beside ties, differed from IEEE division). */
struct DivConst {
    double rhx, rhy, rhz;     /* 1/hx, 1/hy, 1/hz */
    double r12;               /* 1/12 */
    double Dx, Dy, Dz;        /* (tau hy) hz, (tau hx) hz, (tau hx) hy (cell.h:1578-1580) */
    double rDx, rDy, rDz;
};

inline DivConst make_divconst(const Grid &g) {
    DivConst d;
    d.rhx = 1.0 / g.hx;
    d.rhy = 1.0 / g.hy;
    d.rhz = 1.0 / g.hz;
    d.r12 = 1.0 / 12.0;
    d.Dx = g.tau * g.hy * g.hz;
    d.Dy = g.tau * g.hx * g.hz;
    d.Dz = g.tau * g.hx * g.hy;
    d.rDx = 1.0 / d.Dx;
    d.rDy = 1.0 / d.Dy;
    d.rDz = 1.0 / d.Dz;
    return d;
}

/* pow(v, -0.5) (particle.h:73,116): the hardware's estimate (error up to
 * 6e-8) refined by one step of third order to the last bit or so, then by one
 * Newton step whose residual 1 - v r^2 comes from FMAs, exact but for its last
 * rounding.  That rounds correctly except beside ties, as divc does from recip
 * (none of 2*10^7 random v in 1..51 differed from quad precision).  v is 1 + p.p
 * here: no denormals.  15 instructions, where a square root and a reciprocal
 * before the Newton step took about 50. */
__device__ __forceinline__ double pow_m05(double v) {
    const double r0 = __builtin_amdgcn_rsq(v);
    const double e0 = fma(-v * r0, r0, 1.0);
    const double r = fma(r0 * e0, fma(0.375, e0, 0.5), r0);
    const double rr = r * r;
    const double rr_lo = fma(r, r, -rr);
    double e = fma(-v, rr, 1.0);
    e = fma(-v, rr_lo, e);
    return fma(0.5 * r, e, r);
}

__device__ __forceinline__ double divc(double x, double d, double r) {
    double q0 = x * r;
    double e = fma(-q0, d, x);
    return fma(e, r, q0);
}

/* cell.h:1427-1478 Reflect: (x>xm)(x-xm) + (x<0)(xm+x) + (0<x<xm) x.  The
 * select form returns the same bits in every case, including exact 0 and xm
 * (both map to +0) and the signed zeros of the products. */
__device__ __forceinline__ double reflect1(double x, double xm) {
    return x > xm ? x - xm : (x < 0.0 ? xm + x : ((x > 0 && x < xm) ? x : 0.0));
}

template <int BY, int BZ>
__device__ __forceinline__ double interp(const double *F, int n, double sx1, double sy1,
                                         double sz1, double sx, double sy, double sz) {
    /* cell.h:1054-1153 Interpolate3D in its order: t2 + t1 */
    const double *p = F + n;
    double t_ilk = p[0], t_ilk1 = p[1], t_il1k = p[BZ], t_il1k1 = p[BZ + 1];
    double t_i1lk = p[BY * BZ], t_i1lk1 = p[BY * BZ + 1];
    double t_i1l1k = p[BY * BZ + BZ], t_i1l1k1 = p[BY * BZ + BZ + 1];
    double t1 = sx * (sy * (sz * t_ilk + sz1 * t_ilk1) + sy1 * (sz * t_il1k + sz1 * t_il1k1));
    double t2 = sx1 * (sy * (sz * t_i1lk + sz1 * t_i1lk1) + sy1 * (sz * t_i1l1k + sz1 * t_i1l1k1));
    return t2 + t1;
}

/* the same in the differentiable form, from the far-plane weights (the near
 * ones are 1 minus them).  A node of the box is (value, difference to the
 * next node along z), so a z pair is one fused multiply-add, and the y and x
 * pairs follow from their differences: 10 instructions a component, where the
 * eight products of the reference's order took 21. */
template <int BY, int BZ>
__device__ __forceinline__ double interp(const double2 *F, int n, double sx1, double sy1,
                                         double sz1, double, double, double) {
    const double2 *p = F + n;
    const double2 a = p[0], b = p[BZ], c = p[BY * BZ], d = p[BY * BZ + BZ];
    const double z00 = fma(sz1, a.y, a.x), z01 = fma(sz1, b.y, b.x);
    const double z10 = fma(sz1, c.y, c.x), z11 = fma(sz1, d.y, d.x);
    const double y0 = fma(sy1, z01 - z00, z00), y1 = fma(sy1, z11 - z10, z10);
    return fma(sx1, y1 - y0, y0);
}

struct Geo {
    double hx, hy, hz;
    int n0;           /* node of the owner cell in the tile's box */
};

/* GetField (cell.h:1257-1290): tile indices from (x - x0)/h
 * (getCellNumber, getCellNumberCenter: cell.h:527-549), weights from the
 * global x/h (s1..s6_interpolate: cell.h:1193-1236). */
struct GatherIdx {
    int ix, i1x, iy, i1y, iz, i1z;
    double f1[3], f15[3];   /* the weight floors (int)(x/h + 1), (int)(x/h + 1.5) per axis */
    double s1, s2, s3, s4, s5, s6;
    bool ok;          /* every index inside the tile stencil (2..3) */
};

/* the weights of GetField from given floors f1, f15 per axis (the same
 * arithmetic as gather_index): s = f1 - x/h, s' = f15 - 0.5 - x/h */
__device__ __forceinline__ void gather_weights(GatherIdx &G, double xh, double yh, double zh) {
    G.s1 = G.f1[0] - xh;
    G.s2 = G.f15[0] - 0.5 - xh;
    G.s3 = G.f1[1] - yh;
    G.s4 = G.f15[1] - 0.5 - yh;
    G.s5 = G.f1[2] - zh;
    G.s6 = G.f15[2] - 0.5 - zh;
}

__device__ __forceinline__ bool gather_ok(const GatherIdx &G) {
    return (unsigned)((G.ix - 2) | (G.i1x - 2) | (G.iy - 2) | (G.i1y - 2) | (G.iz - 2) |
                      (G.i1z - 2)) <= 1u;
}

__device__ __forceinline__ GatherIdx gather_index(double x, double y, double z, double frx,
                                                  double fry, double frz, const Grid &g,
                                                  const DivConst &dc) {
    GatherIdx G;
    const double xh = divc(x, g.hx, dc.rhx), yh = divc(y, g.hy, dc.rhy),
                 zh = divc(z, g.hz, dc.rhz);
    G.ix = (int)(frx + 1.0) + 1;
    G.i1x = (int)((frx + 1.0) + 1.5);
    G.iy = (int)(fry + 1.0) + 1;
    G.i1y = (int)((fry + 1.0) + 1.5);
    G.iz = (int)(frz + 1.0) + 1;
    G.i1z = (int)((frz + 1.0) + 1.5);
    G.f1[0] = trunc(xh + 1.0);
    G.f15[0] = trunc(xh + 1.5);
    G.f1[1] = trunc(yh + 1.0);
    G.f15[1] = trunc(yh + 1.5);
    G.f1[2] = trunc(zh + 1.0);
    G.f15[2] = trunc(zh + 1.5);
    gather_weights(G, xh, yh, zh);
    G.ok = gather_ok(G);
    return G;
}

/* 1/d for normal d: the hardware's estimate (relative error below 2^-20) and
 * one step of third order.  Within an ulp, the correctly rounded reciprocal in
 * all but 0.2% of cases or fewer; for divc, whose comment says what follows. */
__device__ __forceinline__ double recip(double d) {
    const double r = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

/* Particle::Move (particle.h:160-202) with every intermediate the adjoint
 * needs: pm = p + tau1 E, ps = tau1 pow(pm.pm+1,-1/2), b = ps H,
 * s = pm + pm x b, pp = Cayley rotation of s, p1 = pp + tau1 E,
 * g2 = pow(p1.p1+1,-1/2), x1 = x + tau g2 p1.  FUSED (differentiable form): the
 * rotation multiplied out, (s + (b.s) b + s x b) / (1 + b.b), and fused
 * multiply-adds throughout, about 70 instructions; else the reference's
 * products and sums, 115. */
struct Boris {
    double pm[3], ps, b[3], s[3], sden, p1[3], g2;
};

template <bool FUSED>
__device__ __forceinline__ Boris boris_move(double pu, double pv, double pw, double Ex, double Ey,
                                            double Ez, double Hx, double Hy, double Hz,
                                            double tau1) {
    Boris B;
    if constexpr (FUSED) {
        pu = fma(tau1, Ex, pu);
        pv = fma(tau1, Ey, pv);
        pw = fma(tau1, Ez, pw);
        B.pm[0] = pu;
        B.pm[1] = pv;
        B.pm[2] = pw;
        const double ps = tau1 * pow_m05(fma(pu, pu, fma(pv, pv, fma(pw, pw, 1.0))));
        B.ps = ps;
        const double bx = ps * Hx, by = ps * Hy, bz = ps * Hz;
        B.b[0] = bx;
        B.b[1] = by;
        B.b[2] = bz;
        const double su = fma(pv, bz, fma(-pw, by, pu));
        const double sv = fma(pw, bx, fma(-pu, bz, pv));
        const double sw = fma(pu, by, fma(-pv, bx, pw));
        B.s[0] = su;
        B.s[1] = sv;
        B.s[2] = sw;
        const double bs = fma(bx, su, fma(by, sv, bz * sw));
        const double sden = fma(bx, bx, fma(by, by, fma(bz, bz, 1.0)));
        B.sden = sden;
        const double rden = recip(sden);   /* one reciprocal for the three quotients */
        pu = divc(fma(bs, bx, fma(sv, bz, fma(-sw, by, su))), sden, rden);
        pv = divc(fma(bs, by, fma(sw, bx, fma(-su, bz, sv))), sden, rden);
        pw = divc(fma(bs, bz, fma(su, by, fma(-sv, bx, sw))), sden, rden);
        pu = fma(Ex, tau1, pu);
        pv = fma(Ey, tau1, pv);
        pw = fma(Ez, tau1, pw);
        B.p1[0] = pu;
        B.p1[1] = pv;
        B.p1[2] = pw;
        B.g2 = pow_m05(fma(pu, pu, fma(pv, pv, fma(pw, pw, 1.0))));
    } else {
        pu += tau1 * Ex;
        pv += tau1 * Ey;
        pw += tau1 * Ez;
        B.pm[0] = pu;
        B.pm[1] = pv;
        B.pm[2] = pw;
        double ps = tau1 * pow_m05((pu * pu + pv * pv + pw * pw) * 1. + 1.0);
        B.ps = ps;
        double bx = ps * Hx, by = ps * Hy, bz = ps * Hz;
        B.b[0] = bx;
        B.b[1] = by;
        B.b[2] = bz;
        double su = pu + pv * bz - pw * by;
        double sv = pv + pw * bx - pu * bz;
        double sw = pw + pu * by - pv * bx;
        B.s[0] = su;
        B.s[1] = sv;
        B.s[2] = sw;
        double q1 = bx * bx, q2 = by * by, q3 = bz * bz;
        double q4 = bx * by, q5 = by * bz, q6 = bz * bx;
        double sden = q1 + 1. + q2 + q3;
        B.sden = sden;
        const double rden = recip(sden);   /* one reciprocal for the three quotients */
        double pu1 = divc((q1 + 1.) * su + (q4 + bz) * sv + (q6 - by) * sw, sden, rden);
        double pv1 = divc((q4 - bz) * su + (q2 + 1.) * sv + (q5 + bx) * sw, sden, rden);
        double pw1 = divc((q6 + by) * su + (q5 - bx) * sv + (q3 + 1.) * sw, sden, rden);
        pu = pu1 + Ex * tau1;
        pv = pv1 + Ey * tau1;
        pw = pw1 + Ez * tau1;
        B.p1[0] = pu;
        B.p1[1] = pv;
        B.p1[2] = pw;
        B.g2 = pow_m05(((pu * pu + pv * pv + pw * pw) + 1.0));
    }
    return B;
}

/* x1 = x + tau g2 p1 along one axis */
template <bool FUSED>
__device__ __forceinline__ double advance(double x, double tau, double g2, double p1) {
    return FUSED ? fma(tau * g2, p1, x) : x + tau * (g2 * p1);
}

/* CurrentToMesh (cell.h:1306-1422): tile indices of both ends
 * (getCellNumberCenterCurrent, cell.h:560-566), crossing code
 * m = 4|di| + 2|dl| + |dk|, relay point x2 on the crossed dual-cell faces
 * (getCellTransitAverage, cell.h:600-602); the uncrossed coordinates follow
 * the straight path at parameter sr = num/den (getRatioBasedX, cell.h:617).
 * Coordinates are relative to the owner cell's corner: the differences are
 * exact, and the products lose nothing to the box's extent.  For one crossed
 * axis num and den carry its displacement as a common factor, so one sum over
 * the crossed axes serves every code. */
struct Relay {
    int i1x, i1y, i1z, i2x, i2y, i2z, m;
    double fx, fy, fz, den, sr;
    double x2x, x2y, x2z;
};

/* the relay geometry from given end cells i1 (start) and i2 (end) */
__device__ __forceinline__ Relay relay_from(double x, double y, double z, double x1, double y1,
                                            double z1, const Geo &G, int i1x, int i1y, int i1z,
                                            int i2x, int i2y, int i2z) {
    Relay R;
    R.i1x = i1x;
    R.i1y = i1y;
    R.i1z = i1z;
    R.i2x = i2x;
    R.i2y = i2y;
    R.i2z = i2z;
    int m = 4 * abs(R.i2x - R.i1x) + 2 * abs(R.i2y - R.i1y) + abs(R.i2z - R.i1z);
    if (m > 7) m = 0;
    R.m = m;
    const double dx = x1 - x, dy = y1 - y, dz = z1 - z;
    R.fx = G.hx * ((double)(i1x + i2x) * 0.5 - 2.0);
    R.fy = G.hy * ((double)(i1y + i2y) * 0.5 - 2.0);
    R.fz = G.hz * ((double)(i1z + i2z) * 0.5 - 2.0);
    const double cx = m & 4 ? dx : 0.0, cy = m & 2 ? dy : 0.0, cz = m & 1 ? dz : 0.0;
    const double num = fma(R.fx - x, cx, fma(R.fy - y, cy, (R.fz - z) * cz));
    R.den = fma(cx, cx, fma(cy, cy, cz * cz));
    R.sr = divc(num, R.den, recip(R.den));
    R.x2x = m & 4 ? R.fx : fma(dx, R.sr, x);
    R.x2y = m & 2 ? R.fy : fma(dy, R.sr, y);
    R.x2z = m & 1 ? R.fz : fma(dz, R.sr, z);
    return R;
}

/* the same with the end cells from fr = x/h and t1 = x1/h */
__device__ __forceinline__ Relay relay_point(double x, double y, double z, double x1, double y1,
                                             double z1, double frx, double fry, double frz,
                                             double t1x, double t1y, double t1z, const Geo &G) {
    return relay_from(x, y, z, x1, y1, z1, G, (int)((frx + 1.5) + 1), (int)((fry + 1.5) + 1),
                      (int)((frz + 1.5) + 1), (int)((t1x + 1.5) + 1), (int)((t1y + 1.5) + 1),
                      (int)((t1z + 1.5) + 1));
}

#endif
