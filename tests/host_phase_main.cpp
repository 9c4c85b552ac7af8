// Host check of the fast variant's phase sine and cosine (phase_sincos,
// st_device.h) against long double: prints the worst absolute error over the
// ranges below and exits 1 above the bound given as argument 1.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>

#include "../spin-tracking_amd/csrc/st_device.h"

static double worst = 0.0;

static void check(double x) {
    double s, c;
    st::phase_sincos(x, s, c);
    const double es = (double)fabsl((long double)s - sinl((long double)x));
    const double ec = (double)fabsl((long double)c - cosl((long double)x));
    const double e = fmax(es, ec);
    if (!(e <= worst)) worst = e;
}

int main(int argc, char** argv) {
    const double bound = argc > 1 ? atof(argv[1]) : 0.0;
    unsigned long long u = 12345;
    auto unit = [&]() {
        u = u * 6364136223846793005ull + 1442695040888963407ull;
        return (double)(u >> 11) * 0x1.0p-53;
    };
    // ordinary phases, small ones, and magnitudes up to the reduction's end
    for (int i = 0; i < 400000; ++i) check((unit() - 0.5) * 2.0e6);
    for (int i = 0; i < 100000; ++i) check(ldexp(unit() - 0.5, -(int)(40 * unit())));
    for (int i = 0; i < 400000; ++i) check(ldexp(unit() - 0.5, (int)(45 * unit())));
    // around the multiples of pi/4, where the quadrant changes
    for (int n = -2000; n <= 2000; ++n)
        for (int d = -2; d <= 2; ++d) {
            double x = n * 0.78539816339744830962;
            for (int k = 0; k < (d < 0 ? -d : d); ++k) x = nextafter(x, d < 0 ? -INFINITY : INFINITY);
            check(x);
        }
    printf("phase sincos worst error %.3g\n", worst);
    double s, c;
    st::phase_sincos(INFINITY, s, c);
    if (!isnan(s) || !isnan(c)) return 1;
    st::phase_sincos(NAN, s, c);
    if (!isnan(s) || !isnan(c)) return 1;
    st::phase_sincos(0.0, s, c);
    if (s != 0.0 || c != 1.0) return 1;
    return worst <= bound ? 0 : 1;
}
