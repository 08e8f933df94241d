// The two-lane flux (csrc/gkm_pair.hpp) and its two-lane reverse pass
// (csrc/adj_pair.hpp) against the one-lane forms on the host: the lanes of a face
// are two threads that exchange values where the lanes of a wave would.  Prints
// the largest differences; exit status 1 above argv[1] (flux, of each
// component's largest magnitude) or argv[2] (partials, as adj_math_check).
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>

#include "adj_pair.hpp"

using namespace gkm;

static std::atomic<int> turn{0};
static double box[2];
static void meet(int& phase)
{
    phase += 2;
    turn.fetch_add(1);
    while (turn.load() < phase) std::this_thread::yield();
}
struct ThreadSwap {
    int lane;
    int* phase;
    double operator()(double x) const
    {
        box[lane] = x;
        meet(*phase);
        const double r = box[1 - lane];
        meet(*phase);
        return r;
    }
};
struct Side {
    double s[5], c[5], n[5], t[2][5];
    double S(int q) const { return s[q]; }
    double C(int q) const { return c[q]; }
    double N(int q) const { return n[q]; }
    double T(int k, int q) const { return t[k][q]; }
};
// side's inputs of v (50, rotated frame) in its lane's frame, and back
static int place(int side, int grp) { return (side ? (const int[]){5, 15, 25, 45, 35} : (const int[]){0, 10, 20, 30, 40})[grp]; }
static double sign(int side, int grp, int q) { return side ? (grp == 2 ? (q == 1 ? 1.0 : -1.0) : (q == 1 ? -1.0 : 1.0)) : 1.0; }
static int slot(int side, int q) { return side && (q == 2 || q == 3) ? 5 - q : q; }

int main(int argc, char** argv)
{
    const double gam = 1.4, R = 287.0, T0 = 300.0, dx = 0.1, dt = 2e-4;
    const int N = 1500;
    Gas<double> g{gam, R, 1.0 / 0.7, 1.8e-3, T0, 1e-10, 2};
    const GasK gk = gas_const(g);
    std::mt19937_64 rng(99);
    std::uniform_real_distribution<double> U(-1.0, 1.0);
    std::vector<double> X(50 * N), F(5 * N), G(5 * N), P(50 * N), Q(50 * N), B(5 * N);
    for (int i = 0; i < N; i++) {
        double* v = &X[50 * i];
        const double jump = i % 3 == 0 ? 0.3 : 0.03;
        for (int st = 0; st < 4; st++) {
            const double rho = 1 + jump * U(rng), p = 86100 * (1 + jump * U(rng));
            double m2 = 0;
            v[5 * st] = rho;
            for (int a = 1; a < 4; a++) {
                const double u = 60 + 100 * U(rng);
                v[5 * st + a] = rho * u;
                m2 += u * u;
            }
            v[5 * st + 4] = p / (gam - 1) + 0.5 * rho * m2;
        }
        for (int d = 0; d < 6; d++)
            for (int q = 0; q < 5; q++) v[20 + 5 * d + q] = 0.4 * U(rng) * std::fabs(v[q]);
        for (int q = 0; q < 5; q++) B[5 * i + q] = U(rng) / (q == 4 ? 1e5 : (q == 0 ? 1.0 : 100.0));
    }
    for (int i = 0; i < N; i++) {
        const double* v = &X[50 * i];
        double D[6][5];
        for (int d = 0; d < 6; d++)
            for (int q = 0; q < 5; q++) D[d][q] = v[20 + 5 * d + q];
        gks_flux_tf<double, double>(v, v + 5, v + 10, v + 15, D, collision_time<double>(v, g), dt, dx, g, &F[5 * i]);
        face_flux_vjp(v, dt, dx, g, &B[5 * i], &P[50 * i]);
    }
    auto lane = [&](int side) {
        int phase = 0;
        const ThreadSwap sw{side, &phase};
        for (int i = 0; i < N; i++) {
            const double* v = &X[50 * i];
            double x[50] = {0}, xb[50] = {0}, Fo[5], Fb[5], d[5];
            for (int grp = 0; grp < 5; grp++)
                for (int q = 0; q < 5; q++) x[place(0, grp) + q] = sign(side, grp, q) * v[place(side, grp) + slot(side, q)];
            Side in;
            for (int q = 0; q < 5; q++) {
                in.c[q] = x[q];
                in.s[q] = x[10 + q];
                in.n[q] = x[20 + q];
                in.t[0][q] = x[30 + q];
                in.t[1][q] = x[40 + q];
            }
            const double tau = collision_time_vjp(v, g, d);
            gks_flux_pair(in, tau, dt, dx, gk, sw, Fo);
            if (side == 0)
                for (int q = 0; q < 5; q++) G[5 * i + q] = Fo[q];
            for (int q = 0; q < 5; q++) Fb[q] = (side && q != 1 ? -1.0 : 1.0) * B[5 * i + slot(side, q)];
            double set[AdjPark::kDoubles];
            const AdjPark pk{set, 1};
            for (int i50 = 0; i50 < 45; i50++)
                if (i50 % 10 < 5) pk(AdjIn::place(i50)) = x[i50];
            const double tb = face_flux_vjp_pair(pk, tau, dt, dx, g, Fb, sw, [&](int i50, double y) { xb[i50] = y; });
            for (int q = 0; q < 5; q++) xb[q] = pk(AdjPark::kC + q) + (side == 0 ? tb * d[q] : 0.0);
            for (int grp = 0; grp < 5; grp++)
                for (int q = 0; q < 5; q++)
                    Q[50 * i + place(side, grp) + slot(side, q)] = sign(side, grp, q) * xb[place(0, grp) + q];
        }
    };
    std::thread a(lane, 0), b(lane, 1);
    a.join();
    b.join();
    double top[5] = {0}, ef = 0, ep = 0;
    for (int i = 0; i < N; i++)
        for (int q = 0; q < 5; q++) top[q] = std::fmax(top[q], std::fabs(F[5 * i + q]));
    for (int i = 0; i < N; i++) {
        for (int q = 0; q < 5; q++) ef = std::fmax(ef, std::fabs(F[5 * i + q] - G[5 * i + q]) / top[q]);
        double big = 0, off = 0;
        for (int k = 0; k < 50; k++) {  // partials times the size of their input
            const double s = std::fabs(X[50 * i + k]);
            big = std::fmax(big, std::fabs(P[50 * i + k]) * s);
            off = std::fmax(off, std::fabs(P[50 * i + k] - Q[50 * i + k]) * s);
        }
        ep = std::fmax(ep, off / big);
    }
    std::printf("%d faces: flux %.3e of the largest, partials %.3e of the largest\n", N, ef, ep);
    return ef <= std::atof(argv[1]) && ep <= std::atof(argv[2]) ? 0 : 1;
}
