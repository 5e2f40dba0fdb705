// Checks pairApart (gpuvoxels_amd/csrc/vx3_pair.h), as the kernels compile it, against the
// overlap of pairContact: voxel sizes from 1e-25 to 1e19, lengths within a few units in the last
// place of the contact distance and far from it, positions away from the origin, infinities and
// NaN.  Prints "ok <pairs left out>" when none left out overlaps, else "bad".
#include <cmath>
#include <cstdio>
#include <limits>
#include <random>

#include "../gpuvoxels_amd/csrc/vx3_pair.h"

template <typename real> static long run(unsigned seed) {
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<double> u(0, 1);
    std::normal_distribution<double> g;
    long left = 0;
    const double sizes[] = {1e-25, 1e-20, 1e-15, 1e-6, 1e-2, 1.0, 1e6, 1e18, 1e19};
    for (double size : sizes)
        for (int k = 0; k < 20000; k++) {
            const real nom = (real)(size * (0.5 + 1.5 * u(rng)));
            const float tfi = (float)(0.5 + u(rng)), tfj = (float)(0.5 + u(rng));
            const float dist = vx3::pairDistance<real>(tfi, tfj, nom);
            double d[3] = {g(rng), g(rng), g(rng)};
            const double n = std::sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
            const int kind = k % 3;
            const double far = kind == 0 ? 1 + (int)(17 * u(rng) - 8) * 0x1p-24 : kind == 1 ? 1 + u(rng) * 0x1p-16 : 3 * u(rng);
            real a[3], c[3];
            for (int i = 0; i < 3; i++) {
                a[i] = (real)(k % 2 ? size * 50 * g(rng) : 0.0);
                c[i] = a[i] + (real)(d[i] / n * dist * far);
            }
            for (int bad = 0; bad < 4; bad++) {   // as they are, then one coordinate infinite or NaN
                const real v[4] = {c[1], std::numeric_limits<real>::infinity(), -std::numeric_limits<real>::infinity(),
                                   std::numeric_limits<real>::quiet_NaN()};
                const real y = v[bad];
                const bool apart = vx3::pairApart<real>(a[0], a[1], a[2], c[0], y, c[2], tfi, tfj, nom);
                const float ox = (float)(c[0] - a[0]), oy = (float)(y - a[1]), oz = (float)(c[2] - a[2]);
                const float rel = dist - sqrtf(ox * ox + oy * oy + oz * oz);
                if (apart && rel > 0) { printf("bad: size %g, overlap %g\n", size, (double)rel); return -1; }
                left += apart && bad == 0;
            }
        }
    return left;
}

int main() {
    const long a = run<double>(1), b = run<float>(2);
    if (a >= 0 && b >= 0) printf("ok %ld\n", a < b ? a : b);
    return 0;
}
