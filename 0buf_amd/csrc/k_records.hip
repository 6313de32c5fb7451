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

/* particles of each tile, from the cells' offsets: along z a tile's cells are
 * consecutive */
__global__ __launch_bounds__(PIC_BLOCK) void k_tile_counts(Grid g, TileGeom t, const long *off,
                                                          int *cnt) {
    const unsigned tile = blockIdx.x * PIC_BLOCK + threadIdx.x;
    if (tile >= (unsigned)t.ntiles) return;
    const unsigned a = tile / (unsigned)t.ntz, x = a / (unsigned)t.nty;
    const int I0 = (int)x * TXC, L0 = (int)(a - x * (unsigned)t.nty) * TYC,
              K0 = (int)(tile - a * (unsigned)t.ntz) * TZC;
    const int K1 = K0 + TZC < g.Nz ? K0 + TZC : g.Nz;
    long n = 0;
    for (int i = I0; i < I0 + TXC && i < g.Nx; i++)
        for (int l = L0; l < L0 + TYC && l < g.Ny; l++) {
            const long row = ((long)i * g.Ny + l) * g.Nz;
            n += off[row + K1] - off[row + K0];
        }
    cnt[tile] = (int)n;
}

/* The order in which workgroups take the tiles: by load in classes of a
 * quarter of the mean (a uniform plasma is one class), the fullest first, each
 * class in tile order, dealt to the XCDs in contiguous runs.  A profiled beam's
 * tiles on the axis hold several times the mean; started last, in their place
 * among the others, they left the chip waiting for a few workgroups: the push
 * issued on 51% of its cycles, on 80% in a uniform plasma.  One launch, us, in
 * tile order / fullest first (two launches of 5 us per checkpoint): 128x64x64
 * cells FP64 with a beam of 8 cells' width, push 1199 / 943, particle adjoint
 * 1870 / 1634, arrival 165 / 117; 256x64x64 FP32, push 1436 / 1177, adjoint
 * 2909 / 2518. */
constexpr int ORDER_T = 512, CLASSES = 16;

__global__ __launch_bounds__(ORDER_T) void k_tile_order(int n, const int *cnt, const long *total,
                                                       int *order) {
    __shared__ int at[CLASSES * ORDER_T];   /* per class and thread: its next position */
    __shared__ int part[ORDER_T / 64];
    __shared__ int start[CLASSES + 1];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const float per = *total > 0 ? 4.0f * (float)n / (float)*total : 0.0f;
    auto cls = [&](int c) {
        const float q = (float)c * per + 0.5f;
        return CLASSES - 1 - (q < (float)(CLASSES - 1) ? (int)q : CLASSES - 1);
    };
    const int chunk = (n + ORDER_T - 1) / ORDER_T;
    const int b = min(tid * chunk, n), e = min(b + chunk, n);
    for (int c = 0; c < CLASSES; c++) at[c * ORDER_T + tid] = 0;
    for (int i = b; i < e; i++) at[cls(cnt[i]) * ORDER_T + tid]++;
    __syncthreads();
    /* exclusive scan over all entries, CLASSES consecutive ones a thread */
    int sum = 0;
    for (int k = 0; k < CLASSES; k++) sum += at[tid * CLASSES + k];
    int wave;
    int run = wave_excl_scan(sum, wave);
    if (lane == 0) part[w] = wave;
    __syncthreads();
    for (int k = 0; k < w; k++) run += part[k];
    for (int k = 0; k < CLASSES; k++) {
        const int v = at[tid * CLASSES + k];
        at[tid * CLASSES + k] = run;
        run += v;
    }
    __syncthreads();
    if (tid < CLASSES) start[tid] = at[tid * ORDER_T];
    if (tid == CLASSES) start[CLASSES] = n;
    __syncthreads();
    for (int i = b; i < e; i++) {
        const int c = cls(cnt[i]), s = start[c], m = start[c + 1] - s;
        const int j = at[c * ORDER_T + tid]++ - s;   /* of the class's m tiles */
        const int q = m >> 3, r = m & 7, cut = r * (q + 1);
        const int x = j < cut ? j / (q + 1) : r + (j - cut) / q;
        const int first = j < cut ? x * (q + 1) : cut + (x - r) * q;
        order[s + (j - first) * 8 + x] = i;
    }
}

}  // namespace

void launch_tile_order(const Grid &g, const TileGeom &t, const long *off, int *cnt, int *order,
                       hipStream_t s) {
    const long cells = (long)g.Nx * g.Ny * g.Nz;
    hipLaunchKernelGGL(k_tile_counts, dim3((unsigned)((t.ntiles + PIC_BLOCK - 1) / PIC_BLOCK)),
                       dim3(PIC_BLOCK), 0, s, g, t, off, cnt);
    hipLaunchKernelGGL(k_tile_order, dim3(1), dim3(ORDER_T), 0, s, (int)t.ntiles, cnt, off + cells,
                       order);
}

void launch_record_offsets(const Grid &g, const TileGeom &t, const int *count, int cap,
                           long *tile_sum, unsigned *done, long *off, long room, DevStatus *st,
                           hipStream_t s) {
    const long blocks = std::min((t.ntiles + SCAN_W - 1) / SCAN_W, (long)SCAN_BLOCKS);
    hipLaunchKernelGGL(k_record_offsets, dim3((unsigned)blocks), dim3(SCAN_T), 0, s, g, t, count,
                       cap, tile_sum, done, off, room, st);
}
