// adj_pair.hpp -- reverse-mode derivative of the GKS face flux by two lanes per
// face (no reference counterpart): face_flux_vjp (adj_flux.hpp) split the way
// gks_flux_pair (gkm_pair.hpp) splits the flux.
//
// One lane per face kept both sides' intermediates and 50 input adjoints: with
// all 512 registers of a lane it spilled 2.5 KB, whose traffic was over half of
// its time (0.47 ms per launch at 64^3).  Here each lane takes one side (lane 1 in the mirrored frame: u ->
// -u, tangential directions exchanged), forward and reverse; sums of the forward
// pass that cross between the lanes give the adjoints that cross back the same
// way (the map between the frames is its own transpose), and the adjoints of
// what both lanes hold a copy of (the equilibrium state, the collision time) are
// added over the lanes before they go on.  Terms of the equilibrium state that
// enter with half their weight in each lane do so here too.
//
// A lane's inputs and what a block of the reverse pass does not use wait in its
// column of LDS (AdjPark, 116 KB per workgroup: one per CU, as the registers allow
// anyway), and the largest pieces are basic blocks of their own (adj_one), which
// the register allocator then serves one at a time: as one block the two-lane form
// still spilled 820 B per lane (0.33 ms), split it spills 140 B: 0.16 ms.
#pragma once
#include "adj_flux.hpp"
#include "gkm_pair.hpp"

namespace gkm {

// collision time of a cell and its derivatives: ln tau = ln T / 2 - ln(T + 110.4)
// - ln rho + const, T = (gam - 1)/R (W4 - |W1..3|^2/(2 rho))/rho
__host__ __device__ __forceinline__ double collision_time_vjp(const double W[5], const Gas<double>& g, double d[5])
{
    const double tau = collision_time<double>(W, g);
    const double ir = g_rcp(W[0]), gR = (g.gam - 1.0) / g.R;
    const double k = 0.5 * (W[1] * W[1] + W[2] * W[2] + W[3] * W[3]) * ir;
    const double T = gR * (W[4] - k) * ir;
    const double tT = tau * (g_div(0.5, T) - g_rcp(T + 110.4)) * gR * ir;  // dtau/dT dT/dW4
    d[0] = tT * (2.0 * k - W[4]) * ir - tau * ir;
    d[1] = -tT * W[1] * ir;
    d[2] = -tT * W[2] * ir;
    d[3] = -tT * W[3] * ir;
    d[4] = tT;
    return tau;
}

// Values a lane sets aside while a block that needs its registers runs: its own
// column of `stride` apart doubles (LDS on the device).  fence(): what was put is
// read back from there, not kept.
struct AdjPark {
    // inputs, in the places of AdjIn; then what is set aside
    static constexpr int kC = 0, kS = 5, kN = 10, kT = 15, kWe = 25, kWeb = 30, kF = 35, kE = 40, kEb = 44, kTc = 49,
                         kCb = 52, kP = 55, kDoubles = 58;
    double* p;
    int stride;
    __host__ __device__ __forceinline__ double& operator()(int k) const { return p[k * stride]; }
    __host__ __device__ __forceinline__ void fence() const
    {
#if defined(__HIP_DEVICE_COMPILE__)
        asm volatile("" ::"v"(p) : "memory");  // p escapes here, or the compiler sees that nothing else reaches the memory
        __builtin_amdgcn_sched_barrier(0);
#endif
    }
};
// v as a value the compiler knows nothing of: what is computed from it is computed
// again, not kept from an earlier use
__host__ __device__ __forceinline__ void adj_fresh(double& v)
{
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(v));
#else
    (void)v;
#endif
}
__host__ __device__ __forceinline__ void adj_fresh(Maxw<double>& s)
{
    adj_fresh(s.den);
    adj_fresh(s.u);
    adj_fresh(s.v);
    adj_fresh(s.w);
    adj_fresh(s.lam);
    adj_fresh(s.i2l);
}
// 1, unknown to the compiler: if (adj_one()) { ... } makes a basic block of its
// own, whose registers are allocated apart from what comes before and after
__host__ __device__ __forceinline__ int adj_one()
{
    int one = 1;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+s"(one));
#endif
    return one;
}
// the lane's inputs at side 0's places of face_flux's 50 (cell 0..4, WENO state
// 10..14, normal slope 20..24, slopes along its first and second tangential
// direction 30..34 and 40..44)
struct AdjIn {
    AdjPark pk;
    __host__ __device__ static constexpr int place(int i)
    {
        return i < 10 ? i : (i < 20 ? i - 5 : (i < 30 ? i - 10 : (i < 40 ? i - 15 : i - 20)));
    }
    __host__ __device__ __forceinline__ double operator[](int i) const { return pk(place(i)); }
};

// pk holds the lane's inputs (AdjIn); xbar(i, v) receives their adjoints at the
// same places, but for the cell's, which are left in pk's kC.  tau0: the left
// cell's collision time.  Fbar: the adjoint of the flux in the lane's frame
// (lane 1: -F0, F1, -F3, -F2, -F4 of lane 0's).  Returns the adjoint of tau0.
template <typename SW, typename XB>
__host__ __device__ __forceinline__ double face_flux_vjp_pair(const AdjPark& pk, double tau0, double dt, double dx,
                                                              const Gas<double>& g, double Fbar[5], const SW& sw,
                                                              XB&& xbar)
{
    const AdjIn x{pk};
    auto park = [&](int k, const double v[5]) {
        for (int q = 0; q < 5; q++) pk(k + q) = v[q];
    };
    auto unpark = [&](int k, double v[5]) {
        for (int q = 0; q < 5; q++) v[q] = pk(k + q);
    };
    using namespace vjp;
    const FluxK k{double(g.K + 2), double(g.K + 3), double(g.K + 4), 1.0 / double(g.K + 3), g.inv_prn};
    const double isqpi = 0.5641895835477562869480794515607726;  // 1/sqrt(pi)

    // ---------------- forward
    Maxw<double> S;
    {
        double W[5];
        unpark(AdjPark::kS, W);
        pair_maxw(S, W, g);
    }
    const double pa = 2.0 * S.den * S.i2l, pb = sw(pa);  // rho / lambda of the two sides
    const double taue = tau0 + dt * g_div(::fabs(pa - pb), ::fabs(pa + pb));
    TimeCoefs<double> tc = time_coefs<double>(taue, dt);
    park(AdjPark::kF, Fbar);
    double h[4];
    auto half_start = [&] {
        double s, is;
        f_sqrt_inv(S.lam, s, is);
        const double z = s * S.u, e = f_exp(-z * z);
        const double h0 = half_erfc(-z, e);
        half_tab<4>(S.u, S.i2l, h0, fma(0.5 * isqpi, e * is, S.u * h0), h);
    };
    half_start();
    // the half Maxwellian's <psi> (equilibrium) and <u psi> (p3 flux)
    auto half_moms = [&](double m[5], double n[5]) {
        m[0] = h[0];
        m[1] = h[1];
        m[2] = m[3] = 0.0;
        m[4] = 0.5 * (h[2] + k.kp2 * S.i2l * h[0]);
        n[0] = h[1];
        n[1] = h[2];
        n[2] = n[3] = 0.0;
        n[4] = 0.5 * (h[3] + k.kp2 * S.i2l * h[1]);
    };
    double We[5];
    {
        double m[5], n[5];
        half_moms(m, n);
        tshift(m, S.v, S.w);
        for (int q = 0; q < 5; q++) We[q] = m[q] = S.den * m[q];
        pair_add(We, m, sw);
    }
    pk.fence();
    Maxw<double> E;
    pair_maxw(E, We, g);
    const TState<double> sE{E.u, E.i2l, 2.0 * E.lam};
    const double cBE = tc.gm2 * E.den, cFE = tc.p2 * E.den;
    double Be[5] = {0, 0, 0, 0, 0}, Fs[5] = {0, 0, 0, 0, 0}, by[5] = {0, 0, 0, 0, 0};
    if (adj_one()) {
        SideFwd s;
        side_fwd<0>(S, h[0], h[1], x, E, tc, k, s);
        tshift(s.sy, s.dV, s.dW);
        tshift(s.sz, s.dV, s.dW);
        tshift(s.b, s.dV, s.dW);
        tshift(s.f, s.dV, s.dW);
        for (int q = 0; q < 5; q++) {
            by[q] = s.sy[q];
            Be[q] = s.b[q];
            Fs[q] = s.f[q];
        }
        pair_add(by, s.sz, sw);
    }
    pk.fence();
    // equilibrium half with the cell's normal slope
    double se, ise;
    f_sqrt_inv(E.lam, se, ise);
    const double ze = se * E.u, ee = f_exp(-ze * ze);
    const double hp0 = half_erfc(-ze, ee), ge = 0.5 * isqpi * (ee * ise);
    const double cn = 2.0 * g_rcp(E.den * dx);
    auto normal_fwd = [&](double hh[7], double dn[5], double m[5], double a[5]) {
        half_tab<7>(sE.u, sE.th, hp0, E.u * hp0 + ge, hh);
        for (int q = 0; q < 5; q++) {
            dn[q] = We[q] - pk(AdjPark::kC + q);
            m[q] = dn[q] * cn;
        }
        tunshift(m, E.v, E.w);
        slope_t(m, sE, k.inv_prn, k.kp3, k.ikp3, a);
    };
    {
        double hh[7], dn[5], m[5], a[5], t[5];
        normal_fwd(hh, dn, m, a);
        for (int q = 0; q < 5; q++) t[q] = cBE * a[q];
        mom_u(hh + 1, sE.th, k.kp2, k.kp4, t, Be);
        for (int q = 0; q < 5; q++) t[q] = cFE * a[q];
        mom_u(hh + 2, sE.th, k.kp2, k.kp4, t, Fs);
    }
    pk.fence();
    // E's tangential term along this lane's first direction, its time slope
    double fuE[6], ay[5], aE[5], bE[5], tF[5];
    full_tab<6>(sE.u, sE.th, fuE);
    slope_t(by, sE, k.inv_prn, k.kp3, k.ikp3, ay);
    {
        double t[5];
        for (int q = 0; q < 5; q++) t[q] = cBE * ay[q];
        mom_uvw(fuE, sE.th, k.kp4, t, Be, 2);
        for (int q = 0; q < 5; q++) t[q] *= E.v;
        mom_u(fuE, sE.th, k.kp2, k.kp4, t, Be);
        for (int q = 0; q < 5; q++) t[q] = cFE * ay[q];
        mom_uvw(fuE + 1, sE.th, k.kp4, t, Fs, 2);
        for (int q = 0; q < 5; q++) t[q] = Be[q];
        pair_add(Be, t, sw);
    }
    const double idenE = g_rcp(E.den), c1 = 0.5 * tc.p1 * E.den, cV = cFE * E.v;
    for (int q = 0; q < 5; q++) bE[q] = Be[q] * idenE;
    slope_t(bE, sE, k.inv_prn, k.kp3, k.ikp3, aE);
    for (int q = 0; q < 5; q++) tF[q] = cV * ay[q] + c1 * aE[q];
    mom_u(fuE + 1, sE.th, k.kp2, k.kp4, tF, Fs);

    // ---------------- reverse
    MaxwBar Sb = maxw_bar_zero(), Eb = maxw_bar_zero();
    CoefBar cb{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    double Web[5] = {0, 0, 0, 0, 0};
    double thEb = 0.0, cBEb = 0.0, cFEb = 0.0;
    double Fsb[5], Beb[5], byb[5];
    pk.fence();
    unpark(AdjPark::kF, Fsb);
    tshift_vjp(Fs, E.v, E.w, Fsb, Eb.v, Eb.w);
    {
        double fuEb[6] = {0, 0, 0, 0, 0, 0}, ayb[5], tb[5] = {0, 0, 0, 0, 0}, t[5], aEb[5], bEb[5];
        auto zero = [&](double* v) {
            for (int q = 0; q < 5; q++) v[q] = 0.0;
        };
        mom_u_vjp(fuE + 1, sE.th, k.kp2, k.kp4, tF, Fsb, tb, fuEb + 1, thEb);
        for (int q = 0; q < 5; q++) {
            ayb[q] = cV * tb[q];
            aEb[q] = c1 * tb[q];
        }
        {
            const double cVb = dot5(ay, tb), c1b = 0.5 * dot5(aE, tb);
            Eb.v += cFE * cVb;
            cFEb += E.v * cVb;
            cb.p1 += E.den * c1b;
            Eb.den += tc.p1 * c1b;
        }
        slope_t_vjp(bE, sE, k.inv_prn, k.kp3, k.ikp3, aEb, bEb, Eb.u, thEb, Eb.lam2);
        for (int q = 0; q < 5; q++) Beb[q] = bEb[q] = bEb[q] * idenE;
        Eb.den -= dot5(Be, bEb) * idenE;
        pair_add(Beb, bEb, sw);
        for (int q = 0; q < 5; q++) t[q] = cFE * ay[q];
        zero(tb);
        mom_uvw_vjp(fuE + 1, sE.th, k.kp4, t, Fsb, tb, fuEb + 1, thEb, 2);
        for (int q = 0; q < 5; q++) ayb[q] += cFE * tb[q];
        cFEb += dot5(ay, tb);
        for (int q = 0; q < 5; q++) t[q] = cBE * E.v * ay[q];
        zero(tb);
        mom_u_vjp(fuE, sE.th, k.kp2, k.kp4, t, Beb, tb, fuEb, thEb);
        for (int q = 0; q < 5; q++) ayb[q] += cBE * E.v * tb[q];
        {
            const double cVb = dot5(ay, tb);
            Eb.v += cBE * cVb;
            cBEb += E.v * cVb;
        }
        for (int q = 0; q < 5; q++) t[q] = cBE * ay[q];
        zero(tb);
        mom_uvw_vjp(fuE, sE.th, k.kp4, t, Beb, tb, fuEb, thEb, 2);
        for (int q = 0; q < 5; q++) ayb[q] += cBE * tb[q];
        cBEb += dot5(ay, tb);
        slope_t_vjp(by, sE, k.inv_prn, k.kp3, k.ikp3, ayb, byb, Eb.u, thEb, Eb.lam2);
        tab_vjp<6>(sE.u, sE.th, fuE, fuEb, Eb.u, thEb);
        Eb.u += fuEb[1];
    }
    pk.fence();
    adj_fresh(E);
    if (adj_one()) {   // the equilibrium half with the normal slope
        double hh[7], dn[5], m[5], a[5], t[5], tb[5] = {0, 0, 0, 0, 0}, ab[5], hhb[7] = {0, 0, 0, 0, 0, 0, 0};
        normal_fwd(hh, dn, m, a);
        for (int q = 0; q < 5; q++) t[q] = cFE * a[q];
        mom_u_vjp(hh + 2, sE.th, k.kp2, k.kp4, t, Fsb, tb, hhb + 2, thEb);
        for (int q = 0; q < 5; q++) ab[q] = cFE * tb[q];
        cFEb += dot5(a, tb);
        for (int q = 0; q < 5; q++) {
            t[q] = cBE * a[q];
            tb[q] = 0.0;
        }
        mom_u_vjp(hh + 1, sE.th, k.kp2, k.kp4, t, Beb, tb, hhb + 1, thEb);
        for (int q = 0; q < 5; q++) ab[q] += cBE * tb[q];
        cBEb += dot5(a, tb);
        double mb[5], mc[5];
        for (int q = 0; q < 5; q++) mc[q] = dn[q] * cn;  // the shift's input
        slope_t_vjp(m, sE, k.inv_prn, k.kp3, k.ikp3, ab, mb, Eb.u, thEb, Eb.lam2);
        tunshift_vjp(mc, E.v, E.w, mb, Eb.v, Eb.w);
        Eb.den -= dot5(dn, mb) * cn * idenE;  // cn = 2/(den dx)
        for (int q = 0; q < 5; q++) {
            Web[q] += cn * mb[q];
            pk(AdjPark::kC + q) = -cn * mb[q];
        }
        tab_vjp<7>(sE.u, sE.th, hh, hhb, Eb.u, thEb);
        half_start_vjp(E.u, E.lam, 1.0, hh[0], hhb[0], hhb[1], Eb.u, Eb.lam);
    }
    cb.gm2 += E.den * cBEb;
    cb.p2 += E.den * cFEb;
    Eb.den += tc.gm2 * cBEb + tc.p2 * cFEb;
    double hb[4] = {0, 0, 0, 0};
    // the side block needs every register: what it does not use waits in pk
    park(AdjPark::kWe, We);
    park(AdjPark::kWeb, Web);
    {
        const double e[4] = {E.den, E.u, E.lam, E.i2l}, b[5] = {Eb.den, Eb.u, Eb.th + thEb, Eb.lam, Eb.lam2};
        for (int q = 0; q < 4; q++) pk(AdjPark::kE + q) = e[q];
        park(AdjPark::kEb, b);
        pk(AdjPark::kTc) = tc.p0;
        pk(AdjPark::kTc + 1) = tc.p3;
        pk(AdjPark::kTc + 2) = taue;
        pk(AdjPark::kCb) = cb.gm2;
        pk(AdjPark::kCb + 1) = cb.p1;
        pk(AdjPark::kCb + 2) = cb.p2;
        pk(AdjPark::kP) = pa;
        pk(AdjPark::kP + 1) = pb;
    }
    pk.fence();
    if (adj_one()) {
        {
            double W[5];
            unpark(AdjPark::kS, W);
            pair_maxw(S, W, g);
            half_start();
            tc = time_coefs<double>(pk(AdjPark::kTc + 2), dt);
            unpark(AdjPark::kF, Fsb);
            tshift_T(Fsb, E.v, E.w);
        }
        // the side block; its second tangential sum went into the partner's by
        double szb[5] = {0, 0, 0, 0, 0};
        pair_add(szb, byb, sw);
        side_rev<0>(S, h[0], h[1], x, E, tc, k, Beb, Fsb, byb, szb, Sb, Eb, hb[0], hb[1], cb, xbar);
    }
    pk.fence();
    unpark(AdjPark::kWe, We);
    unpark(AdjPark::kWeb, Web);
    unpark(AdjPark::kF, Fbar);
    E.den = pk(AdjPark::kE);
    E.u = pk(AdjPark::kE + 1);
    E.lam = pk(AdjPark::kE + 2);
    E.i2l = pk(AdjPark::kE + 3);
    Eb.den = pk(AdjPark::kEb);
    Eb.u = pk(AdjPark::kEb + 1);
    Eb.th = pk(AdjPark::kEb + 2);
    Eb.lam = pk(AdjPark::kEb + 3);
    Eb.lam2 = pk(AdjPark::kEb + 4);
    tc.p0 = pk(AdjPark::kTc);
    tc.p3 = pk(AdjPark::kTc + 1);
    const TimeCoefs<Dual> tcd = time_coefs<Dual>(Dual(pk(AdjPark::kTc + 2), 1.0), Dual(dt));
    cb.gm2 = pk(AdjPark::kCb);
    cb.p1 = pk(AdjPark::kCb + 1);
    cb.p2 = pk(AdjPark::kCb + 2);
    thEb = 0.0;
    if (adj_one()) {   // F64 += p0/2 den_e tshift(m0), m0 = (U, f2, 0, 0, (f3 + (K+2) th U)/2)
        const double f2 = E.u * E.u + E.i2l, f3 = E.u * f2 + 2.0 * E.i2l * E.u;
        double m0[5] = {E.u, f2, 0.0, 0.0, 0.5 * (f3 + k.kp2 * E.i2l * E.u)}, m0s[5], m0b[5];
        for (int q = 0; q < 5; q++) m0s[q] = m0[q];
        tshift(m0s, E.v, E.w);
        const double ce = 0.5 * tc.p0 * E.den;
        for (int q = 0; q < 5; q++) m0b[q] = ce * Fbar[q];
        const double ceb = 0.5 * dot5(m0s, Fbar);
        cb.p0 += E.den * ceb;
        Eb.den += tc.p0 * ceb;
        tshift_vjp(m0, E.v, E.w, m0b, Eb.v, Eb.w);
        Eb.u += m0b[0] + 0.5 * k.kp2 * E.i2l * m0b[4];
        double f2b = m0b[1];
        const double f3b = 0.5 * m0b[4];
        thEb += 0.5 * k.kp2 * E.u * m0b[4];
        // f3 = U f2 + 2 th U, f2 = U^2 + th
        Eb.u += (f2 + 2.0 * E.i2l) * f3b;
        f2b += E.u * f3b;
        thEb += 2.0 * E.u * f3b;
        Eb.u += 2.0 * E.u * f2b;
        thEb += f2b;
    }
    Eb.th += thEb;
    {   // the equilibrium state's adjoint is the sum over its two copies
        const double v = Eb.v;
        Eb.den += sw(Eb.den);
        Eb.u -= sw(Eb.u);
        Eb.v += sw(Eb.w);
        Eb.w += sw(v);
        Eb.th += sw(Eb.th);
        Eb.lam += sw(Eb.lam);
        Eb.lam2 += sw(Eb.lam2);
        double t[5];
        for (int q = 0; q < 5; q++) t[q] = Web[q];
        pair_add(Web, t, sw);
        maxw_vjp(We, E, g.gam, Eb, Web);
    }
    if (adj_one()) {   // We = sum of den tshift(m); F64 += p3 den tshift(n)
        double m[5], n[5], ms[5], ns[5], mb[5], nb[5];
        half_moms(m, n);
        for (int q = 0; q < 5; q++) {
            ms[q] = m[q];
            ns[q] = n[q];
        }
        tshift(ms, S.v, S.w);
        tshift(ns, S.v, S.w);
        const double cS = tc.p3 * S.den;
        for (int q = 0; q < 5; q++) {
            mb[q] = S.den * Web[q];
            nb[q] = cS * Fbar[q];
        }
        const double cSb = dot5(ns, Fbar);
        Sb.den += dot5(ms, Web) + tc.p3 * cSb;
        cb.p3 += S.den * cSb;
        tshift_vjp(m, S.v, S.w, mb, Sb.v, Sb.w);
        tshift_vjp(n, S.v, S.w, nb, Sb.v, Sb.w);
        hb[0] += mb[0] + 0.5 * k.kp2 * S.i2l * mb[4];
        hb[1] += mb[1] + nb[0] + 0.5 * k.kp2 * S.i2l * nb[4];
        hb[2] += 0.5 * mb[4] + nb[1];
        hb[3] += 0.5 * nb[4];
        Sb.th += 0.5 * k.kp2 * (h[0] * mb[4] + h[1] * nb[4]);
        tab_vjp<4>(S.u, S.i2l, h, hb, Sb.u, Sb.th);
        half_start_vjp(S.u, S.lam, 1.0, h[0], hb[0], hb[1], Sb.u, Sb.lam);
    }
    // the collision time: taue = tau0 + dt |pa - pb| / |pa + pb|
    double taueb = cb.gm2 * tcd.gm2.d + cb.gm4 * tcd.gm4.d + cb.gm5 * tcd.gm5.d + cb.p0 * tcd.p0.d +
                   cb.p1 * tcd.p1.d + cb.p2 * tcd.p2.d + cb.p3 * tcd.p3.d + cb.p4 * tcd.p4.d + cb.p5 * tcd.p5.d;
    taueb += sw(taueb);
    {
        const double a = pk(AdjPark::kP), b = pk(AdjPark::kP + 1);
        const double A = a - b, B = a + b;
        const double sA = A > 0 ? 1.0 : (A < 0 ? -1.0 : 0.0), sB = B > 0 ? 1.0 : (B < 0 ? -1.0 : 0.0);
        const double fb = dt * taueb, iaB = g_rcp(::fabs(B)), il = g_rcp(S.lam);
        const double pab = fb * sA * iaB - fb * (::fabs(A) * iaB) * sB * iaB;
        Sb.den += pab * il;
        Sb.lam -= pab * a * il;
    }
    {
        double W[5], b[5] = {0, 0, 0, 0, 0};
        unpark(AdjPark::kS, W);
        maxw_vjp(W, S, g.gam, Sb, b);
        for (int q = 0; q < 5; q++) xbar(10 + q, b[q]);
    }
    return taueb;
}

}  // namespace gkm
