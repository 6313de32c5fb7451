/*
 * k_receiver.h -- which cells of an axis take a leaver of the FP64 push.
 *
 * The reference offers a leaver to every cell of its neighbourhood, and a
 * cell r takes it when r h <= v < r h + h (isPointInCell, cell.h:717) with
 * the products and sums rounded: cells may overlap or leave a gap by an ulp.
 *
 * Host and device: the CPU test suite compiles this header on its own.
 */
#ifndef K_RECEIVER_H
#define K_RECEIVER_H

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define PIC_RHD __host__ __device__ __forceinline__
#else
#include <cmath>
#define PIC_RHD inline
#endif

/* the test itself: bit d + 1 is set when the neighbour at d in {-1, 0, 1} of
 * cell i (periodic over n cells) takes v */
PIC_RHD unsigned receivers(double v, double h, int i, int n) {
    unsigned b = 0;
    for (int d = -1; d <= 1; d++) {
        int r = i + d;
        if (r >= n) r -= n; else if (r < 0) r += n;
        const double r0 = (double)r * h;
        if (r0 <= v && v < r0 + h) b |= 1u << (d + 1);
    }
    return b;
}

/* the same from one product with rh = 1/h: away from the cells' faces only
 * the cell trunc(v/h) takes v.  `near` is set where that cannot be told this
 * way: v within 1e-6 h of a face (far more than the rounding of v rh below
 * 2^31 cells), negative, or in no cell of the neighbourhood.  For n >= 3. */
PIC_RHD unsigned receiver(double v, double rh, int i, int n, bool &near) {
    const double t = v * rh, c = trunc(t), f = t - c;
    const bool inner = f > 1e-6 && f < 1.0 - 1e-6 && t < (double)n;
    int d = (inner ? (int)c : i) - i;
    if (d > 1) d -= n; else if (d < -1) d += n;
    if (!inner || d < -1 || d > 1) near = true;
    return 1u << ((d + 1) & 3);
}

#endif
