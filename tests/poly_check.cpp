// Compares the register form of the Sturm root finder with the stack form,
// bit for bit, on the host: prints the number of differing polynomials.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "../povray_amd/csrc/poly_device.h"

using namespace pvx::poly;

template <int N>
static int differs(const double *c) {
    double a[4] = {0, 0, 0, 0}, b[4] = {0, 0, 0, 0};
    const int na = polysolve<N>(N, c, a), nb = polysolve_n<N>(c, b);
    return na != nb || std::memcmp(a, b, na * sizeof(double)) != 0;
}

int main(int argc, char **argv) {
    const int form = std::atoi(argv[1]), n = std::atoi(argv[2]);
    std::mt19937_64 g(7 + form);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    long bad = 0, degenerate = 0, roots = 0;
    for (int it = 0; it < n; it++) {
        double c[5];
        if (form == 0) { // a ray against a torus
            const double R = 0.5 + U(g), r = R * (0.1 + 0.2 * U(g));
            double P[3], D[3], l = 0.0;
            for (int k = 0; k < 3; k++) {
                P[k] = (2.0 * U(g) - 1.0) * (R + 2.0 * r);
                D[k] = 2.0 * U(g) - 1.0;
                l += D[k] * D[k];
            }
            for (int k = 0; k < 3; k++) D[k] /= std::sqrt(l);
            const double k1 = P[0] * P[0] + P[2] * P[2] + P[1] * P[1] - R * R - r * r;
            const double k2 = P[0] * D[0] + P[1] * D[1] + P[2] * D[2];
            c[0] = 1.0;
            c[1] = 4.0 * k2;
            c[2] = 2.0 * (k1 + 2.0 * (k2 * k2 + R * R * D[1] * D[1]));
            c[3] = 4.0 * (k2 * k1 + 2.0 * R * R * P[1] * D[1]);
            c[4] = k1 * k1 + 4.0 * R * R * (P[1] * P[1] - r * r);
        } else if (form == 1) { // coefficients over twelve decades, of both signs
            for (double &x : c) x = (2.0 * U(g) - 1.0) * std::pow(10.0, 12.0 * U(g) - 6.0);
        } else if (form == 2) { // multiples of a quarter, zeros among them: degenerate chains
            for (double &x : c) x = std::round((2.0 * U(g) - 1.0) * 8.0) / 4.0;
            if (c[0] == 0.0) c[0] = 1.0;
        } else if (form == 3) { // roots given: double, triple and negative ones
            const double a = 5.0 * U(g), b = U(g) < 0.5 ? a : 5.0 * U(g);
            const double rs[4] = {a, b, U(g) < 0.3 ? a : 5.0 * U(g), U(g) < 0.3 ? a : -5.0 * U(g)};
            c[0] = 1.0;
            c[1] = c[2] = c[3] = c[4] = 0.0;
            for (int d = 0; d < 4; d++)
                for (int k = d + 1; k > 0; k--) c[k] -= rs[d] * c[k - 1];
        } else { // huge, infinite and undefined coefficients
            for (double &x : c) {
                const double u = U(g);
                x = u < 0.1 ? HUGE_VAL : u < 0.2 ? -HUGE_VAL : u < 0.3 ? NAN : (2.0 * U(g) - 1.0) * (u < 0.6 ? 1e200 : 1.0);
            }
        }
        double v[4];
        const int nr = polysolve_reg<4>(c, v);
        degenerate += nr < 0;
        roots += nr > 0 ? nr : 0;
        bad += differs<4>(c) + differs<3>(c);
    }
    std::printf("%ld %ld %ld\n", bad, degenerate, roots);
    return 0;
}
