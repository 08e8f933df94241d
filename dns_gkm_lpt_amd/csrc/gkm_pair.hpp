// gkm_pair.hpp -- the FP64 GKS interface flux evaluated by two lanes per face.
//
// The flux of gkm_flux.hpp (the reference's flux(), GKMflux.cpp:11-229) keeps
// about 300 registers of FP64 values alive in one lane; at the 256 a lane has
// with two waves per SIMD the sweeps spilled 228-324 B per lane, moved 5-8
// times their algorithmic bytes in spills and kept the VALU 48-58 % busy.
// Here the left and the right side of a face are two neighbouring lanes.
//
//  * Lane 1 works in a mirrored frame: u -> -u, and its two tangential
//    directions exchanged.  The right state's u < 0 half is then a u' > 0
//    half, so both lanes run the same instructions on their own state, its
//    slopes and its cell; the equilibrium state's u > 0 / u < 0 halves and its
//    two tangential directions are split over the lanes the same way.
//  * Vectors that both sides add to cross over by DPP (no LDS): the mirrored
//    partner's moment-like vector m is (m0, -m1, m3, m2, m4) here, its flux the
//    negative of that.  21 values cross per face.
//  * The time slope's p1 term, which belongs to neither side, enters with half
//    its weight in each lane; p0 <u psi>_e is added after the exchange.
//  * gm1 den_e <psi>_e + gm3 We (GKMflux.cpp:185) is zero by the definition of
//    We (gm3 = -gm1): left out.
//
// 1075 VALU instructions per lane against 2030 for a face in one lane, and
// nothing spilled (215-235 VGPRs in the sweeps).  With the difference form of
// WENO (gkm_math.hpp) and the ring of cells (gkm_sweep.hpp), 256^3 x / y / z
// sweep: 2.63 / 2.98 / 3.18 -> 1.98 / 2.01 / 2.13 ms.  Built for three waves per
// SIMD (168 VGPRs) it spills 32-40 registers and the sweeps slow by a fifth.
//
// The building blocks (rest frames, moments, slopes) are gkm_flux.hpp's.  The
// equilibrium state's terms come last, when the side's slopes are dead: 184
// VGPRs for the flux alone against 200 with them first.
#pragma once
#include "gkm_flux.hpp"

namespace gkm {

// the partner lane's value (lanes 2i and 2i + 1 exchange); every lane of the
// wave must be active
struct PairSwap {
    __device__ __forceinline__ double operator()(double x) const
    {
        const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0xB1, 0xF, 0xF, true);  // quad_perm 1,0,3,2
        const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0xB1, 0xF, 0xF, true);
        return __hiloint2double(hi, lo);
    }
};

// m += the partner's moment-like vector
template <typename SW>
__host__ __device__ __forceinline__ void pair_add(double m[5], const double p[5], const SW& sw)
{
    m[0] += sw(p[0]);
    m[1] -= sw(p[1]);
    m[2] += sw(p[3]);
    m[3] += sw(p[2]);
    m[4] += sw(p[4]);
}

// maxw_init for the two-lane forms: 1/(2 lambda) = p/rho from the specific energy
// alone, without the density's way in and out again (two roundings less in the
// pressure, which the half-space moments' difference amplifies)
template <typename G>
__host__ __device__ __forceinline__ void pair_maxw(Maxw<double>& s, const double W[5], const G& g)
{
    s.den = W[0];
    const double ir = g_rcp(W[0]);
    s.u = W[1] * ir;
    s.v = W[2] * ir;
    s.w = W[3] * ir;
    s.i2l = gas_gam1(g) * fma(W[4], ir, -0.5 * (s.u * s.u + s.v * s.v + s.w * s.w));
    s.lam = 0.5 * g_rcp(s.i2l);
}

// Inputs of one side through an accessor (the lane's frame: slot 1 the normal
// momentum towards the lane's u > 0, slots 2 and 3 its first and second
// tangential momentum):
//   in.S(q)    : WENO state of the side     in.C(q)    : the side's cell
//   in.N(q)    : normal slope (x' derivative)
//   in.T(k, q) : k = 0, 1 -> slope along the first / second tangential direction
// tau: collision time of the left cell.  F: the flux in lane 0's frame, valid
// in both lanes up to the mirror (lane 1 holds -F0, F1, -F3, -F2, -F4).
template <typename IN, typename G, typename SW>
__host__ __device__ __forceinline__ void gks_flux_pair(const IN& in, double tau, double dt, double dx,
                                                       const G& g, const SW& sw, double F[5])
{
    using T = double;
    const T isqpi = 0.5641895835477562869480794515607726;  // 1/sqrt(pi)
    const KConst<T> kc = gas_k<T>(g);
    const T kp2 = kc.kp2, kp3 = kc.kp3, kp4 = kc.kp4, ikp3 = kc.ikp3, inv_prn = kc.inv_prn;

    Maxw<T> S;
    {
        T W[5];
#pragma unroll
        for (int q = 0; q < 5; q++) W[q] = in.S(q);
        pair_maxw(S, W, g);
    }
    {   // pressure-jump term of the collision time (GKMflux.cpp:156-157)
        const T pa = T(2) * S.den * S.i2l, pb = sw(pa);  // rho / lambda of the two sides
        tau = tau + dt * g_div(::fabs(pa - pb), ::fabs(pa + pb));
    }
    // half-space u table of the side, entries 0 and 1 (gkm_flux.hpp)
    T h0, h1;
    {
        T s, is;
        f_sqrt_inv(S.lam, s, is);
        const T z = s * S.u, e = f_exp(-z * z);
        h0 = half_erfc(-z, e);
        h1 = fma(T(0.5) * isqpi, e * is, S.u * h0);
    }
    T We[5];
    {
        const T h2 = S.u * h1 + S.i2l * h0;
        T m[5] = {S.den * h0, S.den * h1, 0, 0, S.den * (T(0.5) * (h2 + kp2 * S.i2l * h0))};
        tshift(m, S.v, S.w);
#pragma unroll
        for (int q = 0; q < 5; q++) We[q] = m[q];
        pair_add(We, m, sw);
    }
    Maxw<T> E;
    pair_maxw(E, We, g);
    // time-integration coefficients (GKMflux.cpp:162-167, 197-204)
    const T ex = f_exp(-g_div(dt, tau));
    const T om = T(1) - ex;
    const T igm0 = g_rcp(dt - tau * om);
    const T gm2 = (-dt + T(2) * tau * om - dt * ex) * igm0;
    const T gm5 = tau * om * igm0;
    const T gm45 = (dt * ex - tau * om) * igm0 + gm5;
    const T Pc = tau * om;
    const T Qc = -tau * dt * ex + tau * tau * om;
    const T p0 = dt - Pc;
    const T p1 = T(0.5) * dt * dt - tau * p0;
    const T p2 = -tau * p0 + Qc;
    const T p4 = -Qc - tau * Pc;
    const T p5 = -tau * Pc;

    // Be: den_e B_ (GKMflux.cpp:183-190), Fs: the flux, in E's tangential rest frame
    T Be[5] = {0, 0, 0, 0, 0}, Fs[5] = {0, 0, 0, 0, 0}, by[5];
    const T dV = S.v - E.v, dW = S.w - E.w;

    const TState<T> se{E.u, E.i2l, T(2) * E.lam};
    const T cBe = gm2 * E.den, cFe = p2 * E.den;
    {   // the side's own slopes
        const TState<T> st{S.u, S.i2l, T(2) * S.lam};
        const T iden = g_rcp(S.den);
        T ax[5], ay[5], az[5];
        slope_from_lab(in.N(0) * iden, in.N(1) * iden, in.N(2) * iden, in.N(3) * iden, in.N(4) * iden, S.v, S.w, st,
                       inv_prn, kp3, ikp3, ax);
        slope_from_lab(in.T(0, 0) * iden, in.T(0, 1) * iden, in.T(0, 2) * iden, in.T(0, 3) * iden, in.T(0, 4) * iden,
                       S.v, S.w, st, inv_prn, kp3, ikp3, ay);
        slope_from_lab(in.T(1, 0) * iden, in.T(1, 1) * iden, in.T(1, 2) * iden, in.T(1, 3) * iden, in.T(1, 4) * iden,
                       S.v, S.w, st, inv_prn, kp3, ikp3, az);
        T hu[7];
        half_tab<7>(st.u, st.th, h0, h1, hu);
        // V ay + W az: the lab-frame v and w weights split into rest-frame weight + (V, W)
        T tvw[5];
#pragma unroll
        for (int q = 0; q < 5; q++) tvw[q] = S.v * ay[q] + S.w * az[q];
        // time slope A of the state (GKMflux.cpp:134-151)
        T A[5];
        {
            T fu[6];
            full_tab<6>(st.u, st.th, fu);
            T b[5] = {0, 0, 0, 0, 0};
            mom_u(fu + 1, st.th, kp2, kp4, ax, b);
            mom_uvw(fu, st.th, kp4, ay, b, 2);
            mom_uvw(fu, st.th, kp4, az, b, 3);
            mom_u(fu, st.th, kp2, kp4, tvw, b);
#pragma unroll
            for (int q = 0; q < 5; q++) b[q] = -b[q];
            slope_t(b, st, inv_prn, kp3, ikp3, A);
        }
        // den_e B_ terms (GKMflux.cpp:183-190) and flux terms (GKMflux.cpp:223-228)
        {
            const T cB = gm45 * S.den, cA = gm5 * S.den;
            T b[5] = {0, 0, 0, 0, 0}, c[5];
#pragma unroll
            for (int q = 0; q < 5; q++) c[q] = cB * ax[q];
            mom_u(hu + 1, st.th, kp2, kp4, c, b);
#pragma unroll
            for (int q = 0; q < 5; q++) c[q] = cB * ay[q];
            mom_uvw(hu, st.th, kp4, c, b, 2);
#pragma unroll
            for (int q = 0; q < 5; q++) c[q] = cB * az[q];
            mom_uvw(hu, st.th, kp4, c, b, 3);
#pragma unroll
            for (int q = 0; q < 5; q++) c[q] = cB * tvw[q] + cA * A[q];
            mom_u(hu, st.th, kp2, kp4, c, b);
            tshift(b, dV, dW);
#pragma unroll
            for (int q = 0; q < 5; q++) Be[q] += b[q];
        }
        {
            const T cF = p4 * S.den, cA = p5 * S.den;
            T f[5] = {0, 0, 0, 0, 0}, c[5];
#pragma unroll
            for (int q = 0; q < 5; q++) c[q] = cF * ax[q];
            mom_u(hu + 2, st.th, kp2, kp4, c, f);
#pragma unroll
            for (int q = 0; q < 5; q++) c[q] = cF * ay[q];
            mom_uvw(hu + 1, st.th, kp4, c, f, 2);
#pragma unroll
            for (int q = 0; q < 5; q++) c[q] = cF * az[q];
            mom_uvw(hu + 1, st.th, kp4, c, f, 3);
#pragma unroll
            for (int q = 0; q < 5; q++) c[q] = cF * tvw[q] + cA * A[q];
            mom_u(hu + 1, st.th, kp2, kp4, c, f);
            tshift(f, dV, dW);
#pragma unroll
            for (int q = 0; q < 5; q++) Fs[q] += f[q];
        }
        {   // equilibrium tangential slopes' right-hand sides (GKMflux.cpp:130-133, 141-144):
            // this lane goes on with its first direction, the partner's second one
            T t[5] = {0, 0, 0, 0, 0};
            mom_u(hu, st.th, kp2, kp4, az, t);
            tshift(t, dV, dW);
#pragma unroll
            for (int q = 0; q < 5; q++) by[q] = 0;
            mom_u(hu, st.th, kp2, kp4, ay, by);
            tshift(by, dV, dW);
            pair_add(by, t, sw);
        }
    }
    {   // Euler part: p3 <u psi> of the side's half Maxwellian (GKMflux.cpp:226)
        const T h2 = S.u * h1 + S.i2l * h0, h3 = S.u * h2 + T(2) * S.i2l * h1;
        const T c = Pc * S.den;
        T m[5] = {c * h1, c * h2, 0, 0, c * (T(0.5) * (h3 + kp2 * S.i2l * h1))};
        tshift(m, dV, dW);
#pragma unroll
        for (int q = 0; q < 5; q++) Fs[q] += m[q];
    }
    {   // equilibrium state, normal slope of this side (GKMflux.cpp:115-116, 124-125, 170-171, 210-211)
        T s, is;
        f_sqrt_inv(E.lam, s, is);
        const T z = s * E.u, e = f_exp(-z * z);
        T hp[7];
        {
            const T a0 = half_erfc(-z, e);
            half_tab<7>(se.u, se.th, a0, fma(T(0.5) * isqpi, e * is, E.u * a0), hp);
        }
        const T c = T(2) * g_rcp(E.den * dx);
        T a[5], t[5];
        // We in its own rest frame is den (1, u, 0, 0, (u^2 + (K+3) theta)/2)
        T m[5] = {in.C(0), in.C(1), in.C(2), in.C(3), in.C(4)};
        tunshift(m, E.v, E.w);
        m[0] = (E.den - m[0]) * c;
        m[1] = (E.den * E.u - m[1]) * c;
        m[2] *= -c;
        m[3] *= -c;
        m[4] = (T(0.5) * E.den * (E.u * E.u + kp3 * E.i2l) - m[4]) * c;
        slope_t(m, se, inv_prn, kp3, ikp3, a);
#pragma unroll
        for (int q = 0; q < 5; q++) t[q] = cBe * a[q];
        mom_u(hp + 1, se.th, kp2, kp4, t, Be);
#pragma unroll
        for (int q = 0; q < 5; q++) t[q] = cFe * a[q];
        mom_u(hp + 2, se.th, kp2, kp4, t, Fs);
    }
    {   // equilibrium state: this lane's tangential direction (GKMflux.cpp:148-149, 172-173, 212-213),
        // then the time slope (GKMflux.cpp:183-191) and its p1 term (GKMflux.cpp:225)
        T a[5], t[5], fu[6];
        full_tab<6>(se.u, se.th, fu);
        slope_t(by, se, inv_prn, kp3, ikp3, a);
#pragma unroll
        for (int q = 0; q < 5; q++) t[q] = cBe * a[q];
        mom_uvw(fu, se.th, kp4, t, Be, 2);
#pragma unroll
        for (int q = 0; q < 5; q++) t[q] *= E.v;
        mom_u(fu, se.th, kp2, kp4, t, Be);
#pragma unroll
        for (int q = 0; q < 5; q++) a[q] *= cFe;
        mom_uvw(fu + 1, se.th, kp4, a, Fs, 2);
        T b[5];
#pragma unroll
        for (int q = 0; q < 5; q++) b[q] = Be[q];
        pair_add(b, Be, sw);
        const T iden = g_rcp(E.den);
#pragma unroll
        for (int q = 0; q < 5; q++) b[q] *= iden;
        slope_t(b, se, inv_prn, kp3, ikp3, t);
        const T c1 = T(0.5) * p1 * E.den;
#pragma unroll
        for (int q = 0; q < 5; q++) t[q] = E.v * a[q] + c1 * t[q];
        mom_u(fu + 1, se.th, kp2, kp4, t, Fs);
    }
#pragma unroll
    for (int q = 0; q < 5; q++) F[q] = Fs[q];
    F[0] -= sw(Fs[0]);
    F[1] += sw(Fs[1]);
    F[2] -= sw(Fs[3]);
    F[3] -= sw(Fs[2]);
    F[4] -= sw(Fs[4]);
    {   // p0 <u psi>_e (GKMflux.cpp:225), the largest term: last, so that the others' sums round at their own size
        const T f2 = E.u * E.u + E.i2l, f3 = E.u * f2 + T(2) * E.i2l * E.u;
        const T c = p0 * E.den;
        F[0] += c * E.u;
        F[1] += c * f2;
        F[4] += c * (T(0.5) * (f3 + kp2 * E.i2l * E.u));
    }
    tshift(F, E.v, E.w);
}

}  // namespace gkm
