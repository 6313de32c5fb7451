/* axis_step() against the reference's tests it stands for, Reflect, flyDirection,
 * isPointInCell of the own cell and receivers(): every cell of boxes of several
 * sizes, ends in the cell and its neighbours, past them, at faces, an ulp beside
 * them, across the periodic ends, infinite and NaN.  Wherever axis_step()
 * decides, it must decide the same, the position to the bit; it must decide in
 * the interiors of the cell and its neighbours. */
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

#include "k_receiver.h"

static double reflect(double x, double xm) {
    return x > xm ? x - xm : (x < 0.0 ? xm + x : ((x > 0 && x < xm) ? x : 0.0));
}
static int flies(double v, double v0, double h, int i, int n, double L) {
    return ((v > v0 + h) && (v < v0 + 2 * h)) || ((v < h) && (i == n - 1))
               ? 2
               : ((v < v0) || ((v > L - h) && (i == 0)) ? 0 : 1);
}

int main() {
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    long bad = 0, undecided = 0, tried = 0;
    for (int n : {3, 4, 5, 19, 256, 4096, 100000})
        for (double L : {0.1 * n, 1.0, 3.7, 1e-3 * n}) {
            const double h = L / n;
            for (int k = 0; k < 400; k++) {
                const int i = n <= 400 ? k % n : (k < 8 ? k : k < 16 ? n - 1 - (k - 8) : (int)(U(rng) * n));
                const double x0 = (double)i * h;
                for (int q = 0; q < 60; q++) {
                    const int off = (int)(rng() % 5) - 2;   /* cells -2..2 away, unwrapped */
                    double v = (i + off + U(rng)) * h;
                    bool inner = off >= -1 && off <= 1;
                    if (q >= 40) {
                        inner = false;
                        v = (double)(i + off) * h;
                        if (q % 4 == 1) v = std::nextafter(v, 1e300);
                        if (q % 4 == 2) v = std::nextafter(v, -1e300);
                        if (q % 4 == 3) v = (double)(i + off) * h + h;
                        if (q == 50) v = L;
                        if (q == 51) v = std::numeric_limits<double>::quiet_NaN();
                        if (q == 52) v = std::numeric_limits<double>::infinity();
                        if (q == 53) v = 0.0;
                        if (q == 54) v = 1e300;
                        if (q == 55) v = -1e300;
                    }
                    bool near = false;
                    int d = 0;
                    const double a = axis_step(v, (v - x0) / h, i, n, L, d, near);
                    tried++;
                    const double f = v / h - std::floor(v / h);
                    if (near) {
                        if (inner && f > 1e-5 && f < 1 - 1e-5) undecided++;
                        continue;
                    }
                    const double b = reflect(v, L);
                    const bool own = x0 <= b && b < x0 + h;
                    if (std::memcmp(&a, &b, 8) || flies(b, x0, h, i, n, L) != d + 1 ||
                        receivers(b, h, i, n) != 1u << (d + 1) || own != (d == 0))
                        bad++;
                }
            }
        }
    std::printf("%ld tried, %ld wrong, %ld undecided inside a cell\n", tried, bad, undecided);
    return bad || undecided ? 1 : 0;
}
