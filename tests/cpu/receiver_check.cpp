/* receiver() against receivers(): every cell of boxes of several sizes, values
 * in the cell and its neighbours, at faces, an ulp beside them, across the
 * periodic ends, outside the box, negative, infinite and NaN.  Wherever
 * receiver() decides, it must decide the same; it must decide in the cells'
 * interiors. */
#include <cstdio>
#include <limits>
#include <random>

#include "k_receiver.h"

int main() {
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    long bad = 0, undecided = 0, tried = 0;
    for (int n : {3, 4, 5, 19, 256, 4096, 100000})
        for (double L : {0.1 * n, 1.0, 3.7, 1e-3 * n}) {
            const double h = L / n, rh = 1.0 / h;
            for (int k = 0; k < 400; k++) {
                const int i = n <= 400 ? k % n : (k < 8 ? k : k < 16 ? n - 1 - (k - 8) : (int)(U(rng) * n));
                for (int q = 0; q < 40; q++) {
                    const int r = ((i + (int)(rng() % 5) - 2) % n + n) % n;
                    double v = (r + U(rng)) * h;
                    bool inner = true;
                    if (q >= 20) {
                        inner = false;
                        v = (double)r * h;
                        if (q % 4 == 1) v = std::nextafter(v, 1e300);
                        if (q % 4 == 2) v = std::nextafter(v, -1e300);
                        if (q % 4 == 3) v = (double)r * h + h;
                        if (q == 30) v = -v;
                        if (q == 31) v = std::numeric_limits<double>::quiet_NaN();
                        if (q == 32) v = std::numeric_limits<double>::infinity();
                        if (q == 33) v = L + U(rng) * h;
                        if (q == 34) v = 1e300;
                    }
                    bool near = false;
                    const unsigned a = receivers(v, h, i, n), b = receiver(v, rh, i, n, near);
                    tried++;
                    const double f = v / h - std::floor(v / h);
                    if (near) {
                        if (inner && f > 1e-5 && f < 1 - 1e-5 && a != 0) undecided++;
                    } else if (a != b) {
                        bad++;
                    }
                }
            }
        }
    std::printf("%ld tried, %ld wrong, %ld undecided inside a cell\n", tried, bad, undecided);
    return bad || undecided ? 1 : 0;
}
