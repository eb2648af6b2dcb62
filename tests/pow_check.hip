// Host check of cr_pow's short method (cr_pow_quick) against the full-length one it
// replaces: the same bits wherever it answers, and how often it does not.
#include <cstdint>
#include <cstdio>
#include <cstdlib>

#include "../harm_cool_amd/csrc/harm_phys.hpp"

using namespace harm;

static uint64_t s_state = 0x853C49E6748FEA9Bull;
static uint64_t next()
{
    uint64_t z = (s_state += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
static double unit() { return (next() >> 11) * 0x1.0p-53; }

int main(int argc, char **argv)
{
    const long n = argc > 1 ? atol(argv[1]) : 100000;
    long bad = 0, unsure[5] = {0, 0, 0, 0, 0};
    for (long t = 0; t < n; t++) {
        double x, y;
        switch (t % 5) {
        case 0:  // densities and the adiabatic index of the runs
            x = exp(log(1e-12) * unit());
            y = 13. / 9.;
            break;
        case 1:
            x = exp(log(1e-12) * unit());
            y = (t & 1) ? 4. / 3. - 1. : 5. / 3.;
            break;
        case 2:  // next to 1, where log x is small
            x = 1. + ldexp(2. * unit() - 1., -1 - (int)(next() % 52));
            y = 20. * unit() - 10.;
            break;
        case 3:  // the whole range
            x = exp(1380. * unit() - 690.);
            y = 4. * unit() - 2.;
            break;
        default:  // exact powers and their neighbours
            x = (double)(1 + next() % 4096) * ldexp(1., (int)(next() % 40) - 20);
            y = (double)(next() % 4);
            if (next() & 1) x = nextafter(x, (next() & 1) ? 0. : 1e300);
            if (y == 0.) y = 0.5;
            break;
        }
        if (x == 1. || !(x > 0.)) continue;
        double q;
        if (!cr_pow_quick(x, y, q)) {
            unsure[t % 5]++;
            continue;
        }
        const double w = cr_pow_full(x, y);
        if (q != w) {
            if (bad < 5) printf("mismatch x=%a y=%a full %a quick %a\n", x, y, w, q);
            bad++;
        }
    }
    printf("checked %ld mismatches %ld unsure", n, bad);
    for (int k = 0; k < 5; k++) printf(" %ld", unsure[k]);
    printf("\n");
    return bad != 0 || unsure[0] + unsure[1] > n / 100000;
}
