// flight_log against the long double logarithm: prints the largest error in ulp
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include "flight_log.hpp"
using namespace bte;
static const LogEntry tab[FLIGHT_LOG_N] = FLIGHT_LOG_TABLE;
static double worst = 0., at = 0.;
static void one(double u) {
    const double got = flight_log(tab, u);
    const long double want = logl((long double)u);
    if (want == 0.0L) {
        if (got != 0.) worst = INFINITY;
        return;
    }
    const double w = fabs((double)want);
    const double ulp = nextafter(w, INFINITY) - w;
    const double e = (double)(fabsl((long double)got - want) / ulp);
    if (e > worst) worst = e, at = u;
}
int main(int argc, char** argv) {
    const long n = argc > 1 ? atol(argv[1]) : 200000;
    one(1.0);
    for (int i = 1; i < 2000; i++) one(1.0 - ldexp((double)i, -53)), one(ldexp((double)i, -53));
    for (int k = 0; k < 53; k++)
        for (int i = 0; i <= 2 * FLIGHT_LOG_N; i++) {
            const double e = ldexp(0.5 + i / 512.0, -k);
            one(e);
            one(nextafter(e, 0.));
            if (e < 1.) one(nextafter(e, 1.));
        }
    uint64_t s = 88172645463325252ull;
    for (long i = 0; i < n; i++) {
        s ^= s << 13, s ^= s >> 7, s ^= s << 17;
        const double u = 1.0 - (double)(s >> 11) * 0x1p-53;
        one(u);
        one(1.0 - u * 0.0078125);  // the last interval and its neighbour
        one(u * 0x1p-30);
    }
    printf("%.4f %.17g\n", worst, at);
}
