// calq_far_check.hip -- host-only check (built with --cuda-host-only, run on the
// CPU) that the halvings lbm::calq takes at once (calq_far_halvings) are those
// the loop takes one by one: same count outside the band, same q, same step.
// Boundary links of spheres with radii in [lo, hi], a third of them with the
// node ahead just inside the surface, a third grazing.  Test infrastructure.
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "../mglc_amd/csrc/sphere_geom.hpp"

static unsigned long long rng = 0x9E3779B97F4A7C15ull;
static double uni() {  // splitmix64 -> [0, 1)
    unsigned long long z = (rng += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return (double)((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0);
}

int main(int, char** argv) {
    const double lo = atof(argv[1]), hi = atof(argv[2]);
    long long links = 0, skipped = 0, bad = 0;
    for (long long n = 0; n < 3000000; ++n) {
        const double rad = lo + (hi - lo) * uni();
        const int e[3] = {(int)(3 * uni()) - 1, (int)(3 * uni()) - 1, (int)(3 * uni()) - 1};
        const int ga = e[0] * e[0] + e[1] * e[1] + e[2] * e[2];
        if (ga < 1 || ga > 2) continue;
        // the node ahead at distance t <= rad from the centre, along a random
        // direction (for grazing links: nearly normal to e)
        double d[3] = {uni() - 0.5, uni() - 0.5, uni() - 0.5};
        if (n % 3 == 2) {
            const double along = (d[0] * e[0] + d[1] * e[1] + d[2] * e[2]) / ga * (1.0 - 0.1 * uni());
            for (int a = 0; a < 3; ++a) d[a] -= along * e[a];
        }
        const double len = sqrt(lbm::sphere_dist2(d[0], d[1], d[2]));
        const double depth = n % 3 == 0 ? std::pow(10.0, -12.0 * uni()) : std::min(1.5, rad) * uni();
        if (len < 1e-3) continue;
        double D[3];  // the link's node, relative to the centre
        for (int a = 0; a < 3; ++a) D[a] = d[a] / len * (rad - depth) - e[a];
        const double g0 = lbm::sphere_dist2(D[0], D[1], D[2]) - rad * rad;
        const double gb2 = 2.0 * (e[0] * D[0] + e[1] * D[1] + e[2] * D[2]);
        if (g0 <= 0.0) continue;
        const double band = 2.002e-9 * rad + 1e-12 * (rad + 2.0) * (rad + 2.0);
        ++links;
        double q = 0.5, qt = 0.5;
        const int m = lbm::calq_far_halvings(ga, gb2, g0, band, q, qt);
        skipped += m;
        double p = 0.5, pt = 0.5;
        bool ok = true;
        for (int it = 0; it < m; ++it) {
            const double g = __builtin_fma(__builtin_fma((double)ga, p, gb2), p, g0);
            ok = ok && fabs(g) > band;
            pt = pt / 2.0;
            p += g > 0.0 ? pt : -pt;
        }
        bad += !(ok && p == q && pt == qt);
    }
    printf("links %lld skipped %lld mismatches %lld\n", links, skipped, bad);
    return bad != 0;
}
