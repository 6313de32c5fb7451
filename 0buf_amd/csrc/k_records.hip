/*
 * k_records.hip -- offsets of the compact per-step records of the
 * differentiable form (no reference counterpart): the push writes tile t's
 * pre-step particles, in its flat order, at off[t] + (flat index), so the
 * record holds exactly the particles and not the bucket capacity.
 *
 * Tiles are numbered (tx * nty + ty) * ntz + tz and hold 2 x 4 x 8 cells
 * (z fastest), as in the push kernels.
 */
#include <algorithm>

#include "pic_internal.h"

namespace {

constexpr int TXC = 2, TYC = 4, TZC = 8, C = TXC * TYC * TZC;

/* Particles of each tile (bucket counts capped at the capacity), a wavefront
 * per tile, and their exclusive scan by the workgroup that finishes last, each
 * thread a contiguous run of tiles.  (A thread per tile and a second launch
 * whose thread 0 scanned the 1024 run totals took 24 us at 256 tiles and 54 at
 * 16384.)  Few workgroups: each release and acquire passes through the L2s. */
constexpr int SCAN_T = 1024, SCAN_W = SCAN_T / 64, SCAN_BLOCKS = 256;
static_assert(C == 64, "one cell of the tile per lane");

__device__ __forceinline__ long wave_sum(long v) {
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    return v;
}
/* inclusive scan over the lanes of a wavefront */
__device__ __forceinline__ long wave_scan(long v) {
    const int lane = threadIdx.x & 63;
    for (int d = 1; d < 64; d <<= 1) {
        const long y = __shfl_up(v, d);
        if (lane >= d) v += y;
    }
    return v;
}

__global__ __launch_bounds__(SCAN_T) void k_record_offsets(Grid g, TileGeom t, const int *count,
                                                          int cap, long *sum, unsigned *done,
                                                          long *off, long room, DevStatus *st) {
    __shared__ long part[SCAN_W];
    __shared__ bool last;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (long tile = (long)blockIdx.x * SCAN_W + w; tile < t.ntiles;
         tile += (long)gridDim.x * SCAN_W) {
        const int tz = (int)(tile % t.ntz);
        const int ty = (int)((tile / t.ntz) % t.nty);
        const int tx = (int)(tile / ((long)t.ntz * t.nty));
        const int gi = tx * TXC + lane / (TYC * TZC), gl = ty * TYC + (lane / TZC) % TYC,
                  gk = tz * TZC + lane % TZC;
        long v = 0;
        if (gi < g.Nx && gl < g.Ny && gk < g.Nz) {
            const int n = count[((long)gi * g.Ny + gl) * g.Nz + gk];
            v = n < cap ? n : cap;
        }
        v = wave_sum(v);
        if (lane == 0)
            __hip_atomic_store(&sum[tile], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (tid == 0)
        last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) ==
               gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    const long n = t.ntiles, chunk = (n + SCAN_T - 1) / SCAN_T;
    const long b = tid * chunk < n ? tid * chunk : n, e = b + chunk < n ? b + chunk : n;
    auto at = [&](long i) {
        return __hip_atomic_load(&sum[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    long acc = 0;
    for (long i = b; i < e; i++) acc += at(i);
    const long inc = wave_scan(acc);
    if (lane == 63) part[w] = inc;
    __syncthreads();
    long run = inc - acc;
    for (int k = 0; k < w; k++) run += part[k];
    for (long i = b; i < e; i++) {
        off[i] = run;
        run += at(i);
    }
    if (tid == SCAN_T - 1) {   /* the last run ends at the total */
        off[n] = run;
        if (run > room) atomicOr(&st->flags, (unsigned)PIC_F_RECORD);
    }
    if (tid == 0) *done = 0;
}

/* six arrays of n 4-byte words in one launch (the fields of a step
 * record), blockIdx.y = array */
struct Six {
    const unsigned *src[6];
    unsigned *dst[6];
};
__global__ __launch_bounds__(PIC_BLOCK) void k_copy6(Six a, long n) {
    const unsigned *src = a.src[blockIdx.y];
    unsigned *dst = a.dst[blockIdx.y];
    for (long i = (long)blockIdx.x * PIC_BLOCK + threadIdx.x; i < n;
         i += (long)gridDim.x * PIC_BLOCK)
        dst[i] = src[i];
}

}  // namespace

void launch_copy6(void *const dst[6], const void *const src[6], size_t bytes, hipStream_t s) {
    Six a;
    for (int k = 0; k < 6; k++) {
        a.src[k] = (const unsigned *)src[k];
        a.dst[k] = (unsigned *)dst[k];
    }
    const long n = (long)(bytes / 4);
    long blocks = (n + PIC_BLOCK - 1) / PIC_BLOCK;
    if (blocks > 2048) blocks = 2048;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_copy6, dim3((unsigned)blocks, 6), dim3(PIC_BLOCK), 0, s, a, n);
}

void launch_record_offsets(const Grid &g, const TileGeom &t, const int *count, int cap,
                           long *tile_sum, unsigned *done, long *off, long room, DevStatus *st,
                           hipStream_t s) {
    const long blocks = std::min((t.ntiles + SCAN_W - 1) / SCAN_W, (long)SCAN_BLOCKS);
    hipLaunchKernelGGL(k_record_offsets, dim3((unsigned)blocks), dim3(SCAN_T), 0, s, g, t, count,
                       cap, tile_sum, done, off, room, st);
}
