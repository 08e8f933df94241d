// Errors of the two-lane FP64 flux (csrc/gkm_pair.hpp) and of its own square root
// and exponential against 80-bit values: the oracle's C compiled with `double`
// replaced by long double.  The functions run the device's operations (the
// hardware's reciprocal root is stood in for by an FP32 one).  The lanes of a
// face run in turn, again and again, each reading what the other gave in the
// pass before, until every exchange is settled.
// Prints the figures; exit status 1 if a root is further off than argv[1] or the
// exponential than argv[2] (relative), or a flux component's rms error above the
// one-lane form's.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <omp.h>
#include <random>
#include <vector>

#include "gkm_pair.hpp"

namespace ext {
using std::atan;
using std::erfc;
using std::exp;
using std::fabs;
using std::floor;
using std::fmax;
using std::fmin;
using std::fmod;
using std::modf;
using std::pow;
using std::sqrt;
#define double long double
#include "gkm_oracle.c"
#undef double
}  // namespace ext

using namespace gkm;

// swaps of one lane: what it gives, and what the other gave in its last pass
struct Exchange {
    double *mine, *theirs;
    int* k;
    double operator()(double x) const
    {
        mine[*k] = x;
        return theirs[(*k)++];
    }
};
struct Side {
    double s[5], c[5], n[5], t[2][5];
    double S(int q) const { return s[q]; }
    double C(int q) const { return c[q]; }
    double N(int q) const { return n[q]; }
    double T(int k, int q) const { return t[k][q]; }
};

static void two_lanes(const double* v, double tau, double dt, double dx, const GasK& g, double F[5])
{
    Side in[2];
    for (int side = 0; side < 2; side++)
        for (int q = 0; q < 5; q++) {
            const int p = side && (q == 2 || q == 3) ? 5 - q : q;
            const double m = side && q == 1 ? -1.0 : 1.0;
            in[side].c[q] = m * v[5 * side + p];
            in[side].s[q] = m * v[10 + 5 * side + p];
            in[side].n[q] = (side ? -m : m) * v[20 + 5 * side + p];
            in[side].t[0][q] = m * v[(side ? 45 : 30) + p];
            in[side].t[1][q] = m * v[(side ? 35 : 40) + p];
        }
    double given[2][64] = {};
    for (int pass = 0, n = 1; pass <= n; pass++)
        for (int side = 1; side >= 0; side--) {
            int k = 0;
            double Fo[5];
            gks_flux_pair(in[side], tau, dt, dx, g, Exchange{given[side], given[1 - side], &k}, Fo);
            n = k;
            if (side == 0)
                for (int q = 0; q < 5; q++) F[q] = Fo[q];
        }
}

int main(int, char** argv)
{
    const double root_bound = std::atof(argv[1]), exp_bound = std::atof(argv[2]);
    int bad = 0;
    std::mt19937_64 rng(17);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    double es = 0, ei = 0, ee = 0;
    for (int i = 0; i < 2000000; i++) {
        const double x = std::exp(20.0 * U(rng)), z = i % 2 ? -350.0 * (1.0 + U(rng)) : -std::exp(-12.0 + 18.0 * U(rng));
        double s, is;
        f_sqrt_inv(x, s, is);
        const long double r = sqrtl((long double)x), e = expl((long double)z);
        es = std::fmax(es, (double)fabsl((s - r) / r));
        ei = std::fmax(ei, (double)fabsl(is * r - 1.0L));
        if (z > -700.0) ee = std::fmax(ee, (double)fabsl((f_exp(z) - e) / e));
    }
    std::printf("largest relative errors: root %.3e, inverse root %.3e, exp %.3e\n", es, ei, ee);
    bad |= !(es <= root_bound && ei <= root_bound && ee <= exp_bound);
    bad |= f_exp(-1e300) != 0.0 || f_exp(-INFINITY) != 0.0 || f_exp(0.0) != 1.0;

    // smooth flow at Mach 0.3: of uniform density and pressure (a run's first state), and developed
    const double gam = 1.4, R = 287.0, dx = 0.196, dt = 2e-4;
    Gas<double> g{gam, R, 1.0 / 0.7, 2.0, 300.0, 1e-10, 2};
    const GasK gk = gas_const(g);
    ext::orc_gas og{32, 2, gam, R, 0.7, g.mu0, g.T0, dx, g.eps};
    og.prn = 1.0L / g.inv_prn;
    for (int kind = 0; kind < 2; kind++) {
        long double e2[2][5] = {}, f2[5] = {};
        const int N = 20000;
        for (int i = 0; i < N; i++) {
            double v[50];
            const double rho = 1.0 + kind * 0.05 * U(rng), p = 86100.0 * (1.0 + kind * 0.05 * U(rng));
            double u[3];
            for (double& c : u) c = 100.0 * U(rng);
            for (int st = 0; st < 4; st++) {
                const double j = st < 2 ? 1e-2 : 1e-3;  // cells differ more than the two reconstructions
                const double d = rho * (1.0 + kind * j * U(rng)), pp = p * (1.0 + kind * j * U(rng));
                double k2 = 0;
                v[5 * st] = d;
                for (int a = 0; a < 3; a++) {
                    const double c = u[a] + 100.0 * j * U(rng);
                    v[5 * st + 1 + a] = d * c;
                    k2 += c * c;
                }
                v[5 * st + 4] = pp / (gam - 1) + 0.5 * d * k2;
            }
            for (int d = 0; d < 6; d++)
                for (int q = 0; q < 5; q++)
                    v[20 + 5 * d + q] = (q == 4 ? 86100.0 : q == 0 ? 1.0 : 100.0) * (kind || (q && q < 4) ? 0.3 : 0.0) * U(rng);
            const double tau = collision_time<double>(v, g);
            double F1[5], F2[5];
            double D[6][5];
            std::memcpy(D, v + 20, sizeof(D));
            gks_flux_tf<double, double>(v, v + 5, v + 10, v + 15, D, tau, dt, dx, g, F1);
            two_lanes(v, tau, dt, dx, gk, F2);
            long double x[50], F[5];
            for (int k = 0; k < 50; k++) x[k] = v[k];
            ext::orc_flux(x, x + 5, x + 10, x + 15, x + 20, x + 25, x + 30, x + 35, x + 40, x + 45, tau, dt, dx, &og, F);
            for (int q = 0; q < 5; q++) {
                e2[0][q] += (F1[q] - F[q]) * (F1[q] - F[q]);
                e2[1][q] += (F2[q] - F[q]) * (F2[q] - F[q]);
                f2[q] += F[q] * F[q];
            }
        }
        for (int q = 0; q < 5; q++) {
            const double a = (double)sqrtl(e2[0][q] / f2[q]), b = (double)sqrtl(e2[1][q] / f2[q]);
            std::printf("kind %d component %d: one lane %.3e, two lanes %.3e of the rms flux\n", kind, q, a, b);
            bad |= !(b <= a);
        }
    }
    return bad;
}
