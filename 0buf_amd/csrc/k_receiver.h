/*
 * k_receiver.h -- where a particle of the FP64 push ends along an axis, and
 * which cells take it.
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

/* One axis of a move that ends well inside a cell: v1 = where the straight path
 * from cell i (of n >= 3) ends, t = (v1 - i h)/h.  Returns the position wrapped
 * into [0, L) and d in {-1, 0, 1}, the cell it lies in less i.  Reflect, the fly
 * direction, the test of the own cell and the receivers all follow from d alone
 * there.  `near` is set where they may not: v1 within 1e-6 h of a face (far more
 * than the rounding of i h below 2^31 cells), past the neighbours, or NaN. */
PIC_RHD double axis_step(double v1, double t, int i, int n, double L, int &d, bool &near) {
    const double c = floor(t);
    const bool inner = fabs(t - c - 0.5) < 0.5 - 1e-6 && c >= -1.0 && c <= 1.0;
    if (!inner) near = true;
    d = inner ? (int)c : 0;
    const int r = i + d;
    return v1 + (r >= n ? -L : r < 0 ? L : 0.0);
}

#endif
