/*
 * k_gauss.hip -- diagnostics of the particle state, both forms: the Gauss-law
 * residual div E - rho, the per-cell moments and the per-sort moments, all
 * accumulated in FP64 (rho in fixed point).
 *
 * Every kernel here walks the cells' buckets with groups of CL lanes, one
 * cell per group: consecutive lanes take consecutive slots, so a load is
 * coalesced, and no lane is spent on the empty slots of a bucket.  They are
 * bound by reading the particles: at 67M FP32 particles (256x64x64 cells) the
 * density takes 0.11 ms, the other per-cell moments 0.18-0.3 (1.0 GB; 4.9
 * TB/s is this card's copy rate), the per-sort moments 0.62 (from 1.53 with
 * their accumulators in scratch memory).
 *
 * Gauss law: the charge that the current deposit conserves lives on the
 * cell-centre lattice (centre g at (g - 1/2) h, the reference's getNodeX
 * numbering, cell.h:680-692) with cloud-in-cell weights; E shares the J
 * staggering, so div E at centre g is sum_d (E_d[g] - E_d[g - e_d]) / h_d.
 * The Yee update changes div E by -tau div J and the deposit changes rho by
 * the same amount (discrete continuity), so the residual is constant in time
 * up to round-off.  rho is accumulated in int64 fixed point (2^-40): exact
 * and order-free.
 */
#include "pic_internal.h"

namespace {

constexpr int CL = 16;                      /* lanes per cell */
constexpr int CELLS = PIC_BLOCK / CL;       /* cells per workgroup */

__device__ __forceinline__ int bucket_count(const int *count, int cap, long c) {
    const int n = count[c];
    return n < cap ? n : cap;
}

/* sum over the CL lanes of a group (every lane receives it) */
__device__ __forceinline__ double group_sum(double v) {
    for (int d = CL / 2; d > 0; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

__device__ __forceinline__ int wrap1(int g, int N) {   /* centre index into 1..N */
    int b = (g - 1) % N;
    if (b < 0) b += N;
    return b + 1;
}

__device__ __forceinline__ long long fixd(double v) {
    return (long long)llrint(v * PIC_J_SCALE);
}

/* coordinate d of the particle in slot e of a cell whose index along d is
 * i, in cell units and in length units */
__device__ __forceinline__ double at_cells(const PartPtrs &p, int d, long e, int, double h) {
    return p.p[d][e] / h;
}
__device__ __forceinline__ double at_cells(const PartPtrs32 &p, int d, long e, int i, double) {
    return (double)i + (double)p.p[d][e];
}
__device__ __forceinline__ double at_length(const PartPtrs &p, int d, long e, int, double) {
    return p.p[d][e];
}
__device__ __forceinline__ double at_length(const PartPtrs32 &p, int d, long e, int i, double h) {
    return ((double)i + (double)p.p[d][e]) * h;
}

/* rho, one workgroup per tile of 2 x 4 x 8 cells: the eight contributions of
 * a particle go to the tile's node box in LDS (a particle of cell i touches
 * centres i..i+2), the box to the global array once per node.  As eight
 * global atomics per particle this took 20.3 ms at 67M particles
 * (256x64x64 cells), this way 0.50 ms. */
template <int TX, int TY, int TZ, class P>
__global__ __launch_bounds__(PIC_BLOCK) void k_rho(Grid g, TileGeom t, P p, SpeciesTable sp,
                                                  long long *rho) {
    constexpr int C = TX * TY * TZ, BY = TY + 2, BZ = TZ + 2, NB = (TX + 2) * BY * BZ;
    static_assert(C % CELLS == 0, "each group takes C / CELLS cells");
    __shared__ unsigned long long box[NB];
    __shared__ double sM[PIC_MAX_SLOTS];
    const int tid = threadIdx.x, lane = tid % CL;
    const TileAt at = tile_of_block(t, blockIdx.x);
    const int tx = at.tx, ty = at.ty, tz = at.tz;
    for (int n = tid; n < NB; n += PIC_BLOCK) box[n] = 0;
    if (tid < PIC_MAX_SLOTS) sM[tid] = sp.m[tid];
    __syncthreads();
    for (int k = 0; k < C / CELLS; k++) {
        /* the groups of a wavefront take cells four apart: fewer lanes add
         * into one node */
        const int c = (tid / CL) * (C / CELLS) + k;
        const int ca = c / (TY * TZ), cb = (c / TZ) % TY, cc = c % TZ;
        const int gi = tx * TX + ca, gl = ty * TY + cb, gk = tz * TZ + cc;
        if (gi >= g.Nx || gl >= g.Ny || gk >= g.Nz) continue;
        const long cell = ((long)gi * g.Ny + gl) * g.Nz + gk;
        const int n = bucket_count(p.count, p.cap, cell);
        for (int j = lane; j < n; j += CL) {
            const long e = cell * p.cap + j;
            const double a = sM[p.sp[e]];
            const double ux = at_cells(p, 0, e, gi, g.hx), uy = at_cells(p, 1, e, gl, g.hy),
                         uz = at_cells(p, 2, e, gk, g.hz);
            const double fx = floor(ux + 0.5), fy = floor(uy + 0.5), fz = floor(uz + 0.5);
            const double wx1 = ux + 0.5 - fx, wy1 = uy + 0.5 - fy, wz1 = uz + 0.5 - fz;
            const double wx[2] = {1.0 - wx1, wx1}, wy[2] = {1.0 - wy1, wy1},
                         wz[2] = {1.0 - wz1, wz1};
            const int gx = (int)fx, gy = (int)fy, gz = (int)fz;
            /* a particle outside its cell (a replayed tape keeps it there)
             * may reach past the box */
            const bool in = gx >= gi && gx <= gi + 1 && gy >= gl && gy <= gl + 1 && gz >= gk &&
                            gz <= gk + 1;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int a0 = q >> 2, b0 = (q >> 1) & 1, c0 = q & 1;
                const unsigned long long v =
                    (unsigned long long)fixd(a * wx[a0] * wy[b0] * wz[c0]);
                if (in)
                    atomicAdd(&box[((ca + gx - gi + a0) * BY + cb + gy - gl + b0) * BZ + cc + gz -
                                   gk + c0], v);
                else
                    atomicAdd((unsigned long long *)&rho[(long)wrap1(gx + a0, g.Nx) * g.sx +
                                                         (long)wrap1(gy + b0, g.Ny) * g.sy +
                                                         wrap1(gz + c0, g.Nz)], v);
            }
        }
    }
    __syncthreads();
    for (int n = tid; n < NB; n += PIC_BLOCK) {
        const unsigned long long v = box[n];
        if (v == 0) continue;
        const int u = n / (BY * BZ), w = (n / BZ) % BY, z = n % BZ;
        atomicAdd((unsigned long long *)&rho[(long)wrap1(tx * TX + u, g.Nx) * g.sx +
                                             (long)wrap1(ty * TY + w, g.Ny) * g.sy +
                                             wrap1(tz * TZ + z, g.Nz)], v);
    }
}

/* the residual, and its largest distance from ref (null: none) as the bits
 * of a non-negative double, which order as integers */
template <typename T>
__global__ __launch_bounds__(PIC_BLOCK) void k_gauss(Grid g, const T *Ex, const T *Ey,
                                                    const T *Ez, const long long *rho,
                                                    double *res, const double *ref,
                                                    unsigned long long *drift) {
    const long b = (long)blockIdx.x * PIC_BLOCK + threadIdx.x;
    double far = 0.0;
    if (b < (long)g.Nx * g.Ny * g.Nz) {
        const int i = (int)(b / ((long)g.Ny * g.Nz)) + 1, l = (int)((b / g.Nz) % g.Ny) + 1,
                  k = (int)(b % g.Nz) + 1;
        const long n = (long)i * g.sx + (long)l * g.sy + k;
        const double div = ((double)Ex[n] - (double)Ex[n - g.sx]) / g.hx +
                           ((double)Ey[n] - (double)Ey[n - g.sy]) / g.hy +
                           ((double)Ez[n] - (double)Ez[n - 1]) / g.hz;
        const double r = div - (double)rho[n] * PIC_J_INV;
        res[b] = r;
        if (ref) far = fabs(r - ref[b]);
    }
    if (!ref) return;
    if (!(far > 0.0)) far = 0.0;   /* (a NaN counts as none) */
    for (int d = 32; d > 0; d >>= 1) {
        const double o = __shfl_xor(far, d);
        far = o > far ? o : far;
    }
    /* one address for the whole grid: only the waves that raise it add to it
     * (all of them took 190 us at 1M cells, against 9 without the drift) */
    const unsigned long long bits = (unsigned long long)__double_as_longlong(far);
    if (threadIdx.x % 64 == 0 && bits > __hip_atomic_load(drift, __ATOMIC_RELAXED,
                                                          __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(drift, bits);
}

/* Per-cell particle moments (the reference's diagnostics_operations
 * DENSITY, KINETIC_ENERGY, VELOCITY, CURRENT of particle_types.h:15-16,
 * declared there and never implemented): for one sort, per bulk cell,
 *   DENSITY         sum of the charge weights m (= q n of the cell)
 *   KINETIC_ENERGY  sum of (m / q_m)(gamma - 1), gamma - 1 = p.p / (gamma + 1)
 *   VELOCITY        mean of u = p / gamma (3 components)
 *   CURRENT         sum of m u (3 components)
 * accumulated in FP64 over the cell's bucket.  One lane per cell, each
 * walking a bucket of its own, took 2.0-3.0 ms at 67M FP32 particles
 * (256x64x64 cells): every load of a wavefront fell on 64 lines. */
template <int OP, class P>
__global__ __launch_bounds__(PIC_BLOCK) void k_cell_moments(long ncell, P p, SpeciesTable sp,
                                                            const int *slot_sort, int sort,
                                                            double *out) {
    /* per species slot: the weight of a particle in the sum, 0 for the other
     * sorts */
    __shared__ double sW[PIC_MAX_SLOTS];
    __shared__ int sIn[PIC_MAX_SLOTS];
    const int tid = threadIdx.x;
    if (tid < PIC_MAX_SLOTS) {
        sW[tid] = OP == PIC_KINETIC_ENERGY ? sp.m[tid] / sp.q_m[tid] : sp.m[tid];
        sIn[tid] = slot_sort[tid] == sort;
    }
    __syncthreads();
    const long c = (long)blockIdx.x * CELLS + tid / CL;
    if (c >= ncell) return;
    const int n = bucket_count(p.count, p.cap, c);
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, cnt = 0.0;
    for (int j = tid % CL; j < n; j += CL) {
        const long e = c * p.cap + j;
        const int s = p.sp[e];
        if (!sIn[s]) continue;
        if (OP == PIC_DENSITY) {
            a0 += sW[s];
            continue;
        }
        const double px = p.p[3][e], py = p.p[4][e], pz = p.p[5][e];
        const double gm = sqrt(1.0 + px * px + py * py + pz * pz);
        if (OP == PIC_KINETIC_ENERGY) {
            /* gamma - 1 as p.p / (gamma + 1): no cancellation for slow particles */
            a0 += sW[s] * ((px * px + py * py + pz * pz) / (gm + 1.0));
        } else {
            const double m = OP == PIC_CURRENT ? sW[s] : 1.0;
            a0 += m * (px / gm);
            a1 += m * (py / gm);
            a2 += m * (pz / gm);
            cnt += 1.0;
        }
    }
    a0 = group_sum(a0);
    if (OP >= PIC_VELOCITY) {
        a1 = group_sum(a1);
        a2 = group_sum(a2);
        cnt = group_sum(cnt);
        const double d = OP == PIC_VELOCITY && cnt > 0.0 ? cnt : 1.0;
        if (tid % CL == 0) {
            out[c] = a0 / d;
            out[ncell + c] = a1 / d;
            out[2 * ncell + c] = a2 / d;
        }
    } else if (tid % CL == 0) {
        out[c] = a0;
    }
}

/* FP64 moments per sort: N, sum x, y, z, sum p, sum (m/q_m)(gamma-1),
 * sum |p|.  Each workgroup leaves 27 partial sums. */
template <class P>
__global__ __launch_bounds__(PIC_BLOCK) void k_moments(Grid g, long ncell, P p, SpeciesTable sp,
                                                      const int *slot_sort, double *partials) {
    __shared__ double red[PIC_BLOCK / 64][27];
    __shared__ double sK[PIC_MAX_SLOTS];
    __shared__ int sSort[PIC_MAX_SLOTS];
    const int tid = threadIdx.x;
    if (tid < PIC_MAX_SLOTS) {
        sK[tid] = sp.m[tid] / sp.q_m[tid];
        const int srt = slot_sort[tid];
        sSort[tid] = srt < 0 ? 0 : (srt > 2 ? 2 : srt);
    }
    __syncthreads();
    double acc[27];
#pragma unroll
    for (int k = 0; k < 27; k++) acc[k] = 0.0;
    for (long c = (long)blockIdx.x * CELLS + tid / CL; c < ncell; c += (long)gridDim.x * CELLS) {
        const int n = bucket_count(p.count, p.cap, c);
        const int i = (int)(c / ((long)g.Ny * g.Nz)), l = (int)((c / g.Nz) % g.Ny),
                  k = (int)(c % g.Nz);
        for (int j = tid % CL; j < n; j += CL) {
            const long e = c * p.cap + j;
            const int s = p.sp[e];
            const int srt = sSort[s];
            const double px = p.p[3][e], py = p.p[4][e], pz = p.p[5][e];
            const double gm = sqrt(1.0 + px * px + py * py + pz * pz);
            const double v[9] = {1.0, at_length(p, 0, e, i, g.hx), at_length(p, 1, e, l, g.hy),
                                 at_length(p, 2, e, k, g.hz), px, py, pz, sK[s] * (gm - 1.0),
                                 fabs(px) + fabs(py) + fabs(pz)};
#pragma unroll
            for (int q = 0; q < 9; q++) {
                acc[q] += srt == 0 ? v[q] : 0.0;
                acc[9 + q] += srt == 1 ? v[q] : 0.0;
                acc[18 + q] += srt == 2 ? v[q] : 0.0;
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 27; q++) {
        double v = acc[q];
        for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
        if (tid % 64 == 0) red[tid / 64][q] = v;
    }
    __syncthreads();
    if (tid < 27) {
        double v = red[0][tid];
        for (int w = 1; w < PIC_BLOCK / 64; w++) v += red[w][tid];
        partials[(long)blockIdx.x * 27 + tid] = v;
    }
}

/* the partial sums of every workgroup, a wavefront per moment (27 threads
 * that each walked the partials in turn took 0.24 ms) */
constexpr int FINAL_T = 1024;
__global__ __launch_bounds__(FINAL_T) void k_moments_final(const double *partials, int nblocks,
                                                          double *out27) {
    const int lane = threadIdx.x % 64;
    for (int q = threadIdx.x / 64; q < 27; q += FINAL_T / 64) {
        double v = 0.0;
        for (int b = lane; b < nblocks; b += 64) v += partials[(long)b * 27 + q];
        for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
        if (lane == 0) out27[q] = v;
    }
}

inline unsigned blocks_for(long n, int per) { return (unsigned)((n + per - 1) / per); }

template <class P>
void rho(const Grid &g, P p, SpeciesTable sp, long long *r, hipStream_t s) {
    const TileGeom t = make_tile_geom(g.Nx, g.Ny, g.Nz, false);
    hipLaunchKernelGGL((k_rho<2, 4, 8, P>), dim3((unsigned)t.ntiles), dim3(PIC_BLOCK), 0, s, g, t,
                       p, sp, r);
}

template <class T>
void gauss(const Grid &g, const T *Ex, const T *Ey, const T *Ez, const long long *r, double *res,
           const double *ref, unsigned long long *drift, hipStream_t s) {
    hipLaunchKernelGGL(k_gauss<T>, dim3(blocks_for((long)g.Nx * g.Ny * g.Nz, PIC_BLOCK)),
                       dim3(PIC_BLOCK), 0, s, g, Ex, Ey, Ez, r, res, ref, drift);
}

template <class P>
void cell_moments(long ncell, P p, SpeciesTable sp, const int *slot_sort, int sort, int op,
                  double *out, hipStream_t s) {
    const dim3 grid(blocks_for(ncell, CELLS)), block(PIC_BLOCK);
    switch (op) {
    case PIC_DENSITY:
        hipLaunchKernelGGL((k_cell_moments<PIC_DENSITY, P>), grid, block, 0, s, ncell, p, sp,
                           slot_sort, sort, out);
        break;
    case PIC_KINETIC_ENERGY:
        hipLaunchKernelGGL((k_cell_moments<PIC_KINETIC_ENERGY, P>), grid, block, 0, s, ncell, p,
                           sp, slot_sort, sort, out);
        break;
    case PIC_VELOCITY:
        hipLaunchKernelGGL((k_cell_moments<PIC_VELOCITY, P>), grid, block, 0, s, ncell, p, sp,
                           slot_sort, sort, out);
        break;
    default:
        hipLaunchKernelGGL((k_cell_moments<PIC_CURRENT, P>), grid, block, 0, s, ncell, p, sp,
                           slot_sort, sort, out);
    }
}

template <class P>
void moments(const Grid &g, long ncell, P p, SpeciesTable sp, const int *slot_sort,
             double *partials, int nblocks, double *out27, hipStream_t s) {
    hipLaunchKernelGGL(k_moments<P>, dim3(nblocks), dim3(PIC_BLOCK), 0, s, g, ncell, p, sp,
                       slot_sort, partials);
    hipLaunchKernelGGL(k_moments_final, dim3(1), dim3(FINAL_T), 0, s, partials, nblocks, out27);
}

}  // namespace

void launch_rho64(const Grid &g, PartPtrs p, SpeciesTable sp, long long *r, hipStream_t s) {
    rho(g, p, sp, r, s);
}
void launch_rho32(const Grid &g, PartPtrs32 p, SpeciesTable sp, long long *r, hipStream_t s) {
    rho(g, p, sp, r, s);
}
void launch_gauss64(const Grid &g, FieldPtrs f, const long long *r, double *res,
                    const double *ref, unsigned long long *drift, hipStream_t s) {
    gauss<double>(g, f.f[PIC_EX], f.f[PIC_EY], f.f[PIC_EZ], r, res, ref, drift, s);
}
void launch_gauss32(const Grid &g, FieldPtrs32 f, const long long *r, double *res,
                    const double *ref, unsigned long long *drift, hipStream_t s) {
    gauss<float>(g, f.E[0], f.E[1], f.E[2], r, res, ref, drift, s);
}
void launch_cell_moments64(long ncell, PartPtrs p, SpeciesTable sp, const int *slot_sort, int sort,
                           int op, double *out, hipStream_t s) {
    cell_moments(ncell, p, sp, slot_sort, sort, op, out, s);
}
void launch_cell_moments32(long ncell, PartPtrs32 p, SpeciesTable sp, const int *slot_sort,
                           int sort, int op, double *out, hipStream_t s) {
    cell_moments(ncell, p, sp, slot_sort, sort, op, out, s);
}
void launch_moments(const Grid &g, long ncell, PartPtrs p, SpeciesTable sp, const int *slot_sort,
                    double *partials, int nblocks, double *out27, hipStream_t s) {
    moments(g, ncell, p, sp, slot_sort, partials, nblocks, out27, s);
}
void launch_moments32(const Grid &g, long ncell, PartPtrs32 p, SpeciesTable sp,
                      const int *slot_sort, double *partials, int nblocks, double *out27,
                      hipStream_t s) {
    moments(g, ncell, p, sp, slot_sort, partials, nblocks, out27, s);
}
