// Host-side check of the entry points that the kernels call for an excluded-volume pair (energy alone,
// forces alone) against the combined form whose rounding exvol_fast_check.cpp measures: the FP64 path's
// values and flags are the same bit for bit. Prints "<pairs> <deferred> <mismatches>".
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

using std::atan;
using std::atan2;
using std::fabs;
using std::sqrt;

#include "../../picgo_amd/csrc/mdn_terms.h"

using namespace mdn;

int main() {
    std::mt19937_64 rng(41);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    int n = 0, deferred = 0, bad = 0;
    for (int k = 0; k < 60000; k++) {
        // general pairs, pairs in one plane (every third) and parallel ones (every seventh)
        const double z = k % 3 == 0 ? 0.0 : 60.0 * U(rng) - 30.0;
        const D3 a{500.0, 500.0, 500.0}, b{500.0 + 100.0 * U(rng) + 8.0, 500.0 + 40.0 * U(rng), 500.0};
        const D3 c{470.0 + 60.0 * U(rng), 470.0 + 90.0 * U(rng), 500.0 + z};
        const D3 d = k % 7 == 0 ? D3{c.x + (b.x - a.x), c.y + (b.y - a.y), c.z}
                                : D3{c.x + 100.0 * U(rng), c.y + 60.0 * U(rng) - 30.0, 500.0 + (k % 3 == 0 ? 0.0 : z + 20.0 * U(rng))};
        D3 f1[4], f2[4];
        int d1 = 0, d2 = 0;
        bool ok1 = true;
        const double u1 = exvol_energy_forces<double>(a, b, c, d, 1e5, &d1, &ok1, f1);
        const double u2 = exvol_energy<double>(a, b, c, d, 1e5, &d2);
        const bool ok2 = exvol_forces<double>(a, b, c, d, 1e5, f2);
        n++;
        deferred += d1;
        bad += d1 != d2 || ok1 != ok2 || std::memcmp(&u1, &u2, sizeof u1) != 0 || (ok1 && std::memcmp(f1, f2, sizeof f1) != 0);
    }
    std::printf("%d %d %d\n", n, deferred, bad);
    return 0;
}
