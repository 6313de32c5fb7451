/*
 * k_arrive.h -- arrival of the departed particles, FP64 form: the
 * receiving side of the reference's migration (GPU_ArrangeFlights /
 * Cell::Insert, kernels.cu:316-370), where each leaver joins the bucket of
 * the cell that accepts it.
 *
 * One workgroup per source tile, a leaver per thread, in rounds of PIC_BLOCK.
 * A record carries the destination cell twice: as a bulk cell index (dest)
 * and as an index into the tile's halo box of (TX+2) x (TY+2) x (TZ+2) cells.
 * Leavers bound for the same cell are counted in LDS first, so each
 * destination cell costs one global atomic per round instead of one per
 * particle (the beam axis of a skewed workload sends tens of particles per
 * step into the same cells); then every leaver takes base + rank as its slot.
 * A slot past the bucket capacity is kept in the record for the regrow path
 * and raises PIC_F_BUCKET_OVERFLOW.  A record whose halo index or destination
 * cell lies out of range is not placed and raises PIC_F_QUEUE_CORRUPT.  Bound
 * by its scattered writes, seven arrays per arrival.
 */
#ifndef K_ARRIVE_H
#define K_ARRIVE_H

#include "k_fold.h"
#include "k_queue_key.h"
#include "pic_internal.h"

/* workgroups [0, tiles): the arrivals of one tile each (tiles: all, or 0);
 * [tiles, fold_end): the periodic fold of the current; those behind them: where
 * the current still is fixed point, its conversion at the nodes without a fold
 * (as a launch of its own before the fold the conversion took 5 us of a small
 * step) */
template <int TX, int TY, int TZ, class JT>
__global__ __launch_bounds__(PIC_BLOCK) void k_arrive_fold(Grid g, TileGeom t, PartPtrs p,
                                                           QueuePtrs q, DevStatus *st,
                                                           FoldJ<JT> f, unsigned tiles,
                                                           unsigned fold_end) {
    if constexpr (std::is_floating_point_v<JT>) {
        if (blockIdx.x >= fold_end) {
            convert_inner(g, f, (blockIdx.x - fold_end) * PIC_BLOCK + threadIdx.x);
            return;
        }
    }
    if (blockIdx.x >= tiles) {
        fold_class(g, f, (blockIdx.x - tiles) * PIC_BLOCK + threadIdx.x);
        return;
    }
    constexpr int BY = TY + 2, BZ = TZ + 2, NH = (TX + 2) * BY * BZ;
    __shared__ int hcnt[NH];
    __shared__ int hbase[NH];
    const TileAt at = tile_of_block(t, blockIdx.x);
    const long tile = at.tile;
    const int tx = at.tx, ty = at.ty, tz = at.tz;
    const int tid = threadIdx.x;
    int n = q.count[tile];
    n = n < q.qcap ? n : q.qcap;
    Leaver64 *const Q = q.e + tile * (long)q.qcap;
    const long ncell = (long)g.Nx * g.Ny * g.Nz;
    bool bad = false, over = false;
    for (int j0 = 0; j0 < n; j0 += PIC_BLOCK) {
        const int j = j0 + tid;
        Leaver64 r;
        int h = -1, rank = 0;
        if (j < n) r = Q[j];
        for (int k = tid; k < NH; k += PIC_BLOCK) hcnt[k] = 0;
        __syncthreads();
        /* rank of each leaver among the round's leavers for the same cell; a
         * record whose halo index or cell lies out of range is refused */
        if (j < n) {
            h = r.where >> 8;
            if (arrival_entry_ok(h, NH, (long)r.dest, ncell)) {
                rank = atomicAdd(&hcnt[h], 1);
            } else {
                h = -1;
                bad = true;
            }
        }
        __syncthreads();
        /* one claim per destination cell on its bucket count */
        for (int k = tid; k < NH; k += PIC_BLOCK) {
            const int c = hcnt[k];
            if (c == 0) continue;
            int gx = tx * TX - 1 + k / (BY * BZ), gy = ty * TY - 1 + (k / BZ) % BY,
                gz = tz * TZ - 1 + k % BZ;
            if (gx < 0) gx += g.Nx; else if (gx >= g.Nx) gx -= g.Nx;
            if (gy < 0) gy += g.Ny; else if (gy >= g.Ny) gy -= g.Ny;
            if (gz < 0) gz += g.Nz; else if (gz >= g.Nz) gz -= g.Nz;
            hbase[k] = atomicAdd(&p.count[((long)gx * g.Ny + gy) * g.Nz + gz], c);
        }
        __syncthreads();
        if (h >= 0) {
            const int slot = hbase[h] + rank;
            if (slot >= p.cap) {
                Q[j].slot = slot;
                over = true;
            } else {
                const long to = (long)r.dest * p.cap + slot;
                p.p[0][to] = r.xy.x;
                p.p[1][to] = r.xy.y;
                p.p[2][to] = r.zu.x;
                p.p[3][to] = r.zu.y;
                p.p[4][to] = r.vw.x;
                p.p[5][to] = r.vw.y;
                p.sp[to] = (unsigned char)(r.where & 255);
                if (p.id) p.id[to] = r.id;
            }
        }
        __syncthreads();   /* the counts and claims are read above */
    }
    if (over) atomicOr(&st->flags, (unsigned)PIC_F_BUCKET_OVERFLOW);
    if (bad) atomicOr(&st->flags, (unsigned)PIC_F_QUEUE_CORRUPT);
}

#endif
