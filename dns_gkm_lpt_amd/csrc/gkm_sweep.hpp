// gkm_sweep.hpp -- device code of the fused sweep (one workgroup's work) and of
// the CFL reductions, shared by the per-launch kernels (gkm_kernels.hip) and
// the persistent ensemble step (ens_persist.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "gkm_kernels.hpp"
#include "gkm_pair.hpp"

namespace gkm {

__device__ __forceinline__ int wrapi(int x, int n) { return x < 0 ? x + n : (x >= n ? x - n : x); }

// physical strides: y -> nc*nc, x -> nc, z -> 1.
// DIR 0 (x sweep): n = x, a = y, b = z.   DWy pairs with a, DWz with b.
// DIR 1 (y sweep): n = y, a = x, b = z.
// DIR 2 (z sweep): n = z, a = x, b = y (the reference's tangential pairing
//                  of derivsZ, update.cpp:402-455, kept as is).
template <int DIR>
__device__ __forceinline__ long cell_index(int cn, int ca, int cb, int nc)
{
    if (DIR == 0) return ((long)ca * nc + cn) * nc + cb;
    if (DIR == 1) return ((long)cn * nc + ca) * nc + cb;
    return ((long)cb * nc + ca) * nc + cn;
}

// Lines of the plus-shaped set a workgroup reconstructs: the CA x CB interior
// lines plus one line beyond each tangential edge (no corners).
template <int CA, int CB>
struct Lines {
    static constexpr int L = CA * CB + 2 * CA + 2 * CB;
    __device__ static __forceinline__ int id(int ia, int ib)
    {
        if (ia < 0) return CA * CB + ib;
        if (ia >= CA) return CA * CB + CB + ib;
        if (ib < 0) return CA * CB + 2 * CB + ia;
        if (ib >= CB) return CA * CB + 2 * CB + CA + ia;
        return ia * CB + ib;
    }
    __device__ static __forceinline__ void coords(int l, int& ia, int& ib)
    {
        if (l < CA * CB) { ia = l / CB; ib = l % CB; return; }
        l -= CA * CB;
        if (l < CB) { ia = -1; ib = l; return; }
        l -= CB;
        if (l < CB) { ia = CA; ib = l; return; }
        l -= CB;
        if (l < CA) { ia = l; ib = -1; return; }
        l -= CA;
        ia = l;
        ib = CB;
    }
};

// LDS layout of the WENO states (10 values per face and line) and of the face
// fluxes (5 values per face slot and interior line).  The fastest thread index
// is contiguous: the tangential line for the x and y sweeps, the face for the z
// sweep (whose lines are short and whose faces are consecutive in memory).
template <int DIR, int CN, int L>
__device__ __forceinline__ int sw_at(int v, int tn, int l)
{
    return DIR == 2 ? (v * L + l) * CN + tn : (v * CN + tn) * L + l;
}
template <int DIR, int CN, int NL>
__device__ __forceinline__ int sf_at(int q, int slot, int lc)
{
    return DIR == 2 ? (q * NL + lc) * (CN + 1) + slot : (q * (CN + 1) + slot) * NL + lc;
}

// FP64: a face's place in a chunk's fluxes
template <int DIR, int CN, int NL>
__device__ __forceinline__ int pf_at(int tn, int lc)
{
    return DIR == 2 ? lc * CN + tn : tn * NL + lc;
}

// Flux inputs of one face, read where the flux uses them: cell states from the
// (cached) state array, WENO states and their tangential differences from LDS.
// q is the rotated-frame slot (normal momentum in slot 1; update.cpp:361-398, 461-497).
template <int DIR, int CN, int L>
struct SweepIn {
    const double* __restrict__ W;
    long plane, iL, iR;
    const double* s;
    int tn, lc, l_am, l_ap, l_bm, l_bp;
    double two_idx, half_idx;
    __device__ static int phys(int q)
    {
        constexpr int sw = DIR == 1 ? 2 : 3;
        return DIR == 0 ? q : (q == 1 ? sw : (q == sw ? 1 : q));
    }
    __device__ double at(int v, int l) const { return s[sw_at<DIR, CN, L>(v, tn, l)]; }
    __device__ double WL(int q) const { return W[phys(q) * plane + iL]; }
    __device__ double WR(int q) const { return W[phys(q) * plane + iR]; }
    __device__ double Wl(int q) const { return at(phys(q), lc); }
    __device__ double Wr(int q) const { return at(5 + phys(q), lc); }
    __device__ double D(int d, int q) const
    {
        const int p = phys(q);
        switch (d) {
        case 0: return (at(p, lc) - WL(q)) * two_idx;                 // DWxl
        case 1: return (WR(q) - at(5 + p, lc)) * two_idx;             // DWxr
        case 2: return (at(p, l_ap) - at(p, l_am)) * half_idx;        // DWyl
        case 3: return (at(5 + p, l_ap) - at(5 + p, l_am)) * half_idx;  // DWyr
        case 4: return (at(p, l_bp) - at(p, l_bm)) * half_idx;        // DWzl
        default: return (at(5 + p, l_bp) - at(5 + p, l_bm)) * half_idx;  // DWzr
        }
    }
};

// LDS doubles of one tile variant: WENO states (10 per face and line) and
// face fluxes (5 per face slot and interior line)
template <int DIR, int V, bool MIX>
constexpr int sweep_lds_doubles()
{
    constexpr int CN = Tile<DIR, V, MIX>::CN, CA = Tile<DIR, V, MIX>::CA, CB = Tile<DIR, V, MIX>::CB;
    constexpr int L = Lines<CA, CB>::L;
    // mixed: WENO states, face fluxes with the face before the chunk; FP64: the
    // ring of cells, WENO states, face fluxes of two chunks
    return MIX ? 10 * CN * L + 5 * (CN + 1) * CA * CB : 6 * (CN + 5) * L + 10 * CN * L + 10 * CN * CA * CB;
}
constexpr int max3(int a, int b, int c) { return a > b ? (a > c ? a : c) : (b > c ? b : c); }
template <int DIR, bool MIX>
constexpr int sweep_lds_max()
{
    return max3(sweep_lds_doubles<DIR, 0, MIX>(), sweep_lds_doubles<DIR, 1, MIX>(), sweep_lds_doubles<DIR, 2, MIX>());
}
template <bool MIX>
constexpr int kSweepLdsMax = max3(sweep_lds_max<0, MIX>(), sweep_lds_max<1, MIX>(), sweep_lds_max<2, MIX>());

// workgroup -> pencil corner (a0, b0) and segment s of one grid (member).
// FACES: a pencil that would reach past the grid is moved back into it; it takes
// some lines of its neighbour a second time, to the same values.
template <int DIR, int CA, int CB, bool GEN, bool FACES = false>
__device__ __forceinline__ void sweep_pencil(const SweepArgs& p, int bid, int nblk, bool remap, int& a0, int& b0, int& s)
{
    const int nc = p.nc;
    // workgroup -> (pencil, segment); XCD-aware: the hardware deals workgroups
    // round-robin over the 8 XCDs, so give each XCD a contiguous range of pencils.
    if (remap && (nblk & 7) == 0) bid = (bid & 7) * (nblk >> 3) + (bid >> 3);
    s = bid % p.nseg;
    const int pencil = bid / p.nseg;
    const int npb = GEN || FACES ? (nc + CB - 1) / CB : nc / CB;  // pencils across b; with GEN the last may reach past nc
    // z sweep on an exact grid: pencils in 8 x 8 patches, so that the ~64
    // workgroups an XCD runs at once cover a square of lines whose tangential
    // edge lines are mostly interior lines of the same patch, read once into
    // that XCD's L2 (the row order re-read the x edge lines of every strip;
    // 512^3: z sweep 19.55 -> 19.22 ms mixed, 25.44 -> 24.79 ms FP64).  The
    // x and y sweeps keep the row order, which measured faster for them.
    int pa, pb;
    if (DIR == 2 && !GEN && !FACES && (npb & 7) == 0 && ((nc / CA) & 7) == 0) {
        const int t = pencil >> 6, w = pencil & 63, tpb = npb >> 3;
        pa = (t / tpb) * 8 + (w >> 3);
        pb = (t % tpb) * 8 + (w & 7);
    } else {
        pa = pencil / npb;
        pb = pencil % npb;
    }
    a0 = pa * CA;
    b0 = pb * CB;
    if (FACES) {
        a0 = a0 < nc - CA ? a0 : nc - CA;
        b0 = b0 < nc - CB ? b0 : nc - CB;
    }
}

// thread -> face of the chunk: the fastest index is the one contiguous in
// memory (the line for the x and y sweeps, the face for the z sweep)
template <int DIR, int CN, int CA, int CB>
__device__ __forceinline__ void sweep_face(int f, int& tn, int& ta, int& tb)
{
    if (DIR == 2) {
        tn = f % CN;
        tb = (f / CN) % CB;
        ta = f / (CN * CB);
    } else {
        tb = f % CB;
        ta = (f / CB) % CA;
        tn = f / (CA * CB);
    }
}

// The FP64 sweep's flux takes a face's two sides in two lanes, the right one in
// a mirrored frame (gkm_pair.hpp): its WENO states are kept in LDS in the frame
// their lane works in, so that both lanes read slot q at the same offset.
// pair_var: the state variable in slot q of a side (normal momentum first).
template <int DIR>
__host__ __device__ constexpr int pair_var(int side, int q)
{
    constexpr int sw = DIR == 0 ? 1 : (DIR == 1 ? 2 : 3);  // the normal momentum; its place holds rho u
    const int k = side && (q == 2 || q == 3) ? 5 - q : q;
    return k == 1 ? sw : (k == sw ? 1 : k);
}

// its inverse: the slot of state variable v on a side
template <int DIR>
__host__ __device__ constexpr int pair_slot(int side, int v)
{
    for (int q = 0; q < 5; q++)
        if (pair_var<DIR>(side, q) == v) return q;
    return -1;
}

// Mixed: WENO states of every (face, line) of a chunk into sW, by NT threads.
// In the x and y sweeps with an even face count a thread takes two neighbouring
// faces of a line: their stencils share five of seven cells, loaded and turned
// into temperatures once; each face's reconstruction is the same arithmetic as
// a face alone (512^3, 4 x 4 x 16 and 2 x 8 x 16 tiles: x 15.66 -> 14.45 ms,
// y 17.17 -> 16.42 ms).  The z sweep keeps one face per thread: with pairs,
// neighbouring lanes read cells two apart along z and it slowed (19.25 ->
// 20.16 ms); its temperatures are formed after all its loads (formed one by one
// with them, as the pairs' are, the z sweep takes 217 us instead of 209 at 100^3 and
// 692 instead of 672 at 160^3).
template <int DIR, int CN, int CA, int CB, int NT>
__device__ __forceinline__ void weno_chunk(const SweepArgs& p, int n0, int a0, int b0, int tid, double* sW)
{
    using LN = Lines<CA, CB>;
    constexpr int L = LN::L;
    const int nc = p.nc;
    const long plane = p.plane;
    const double* __restrict__ W = p.W;
    constexpr int NH = DIR != 2 && CN % 2 == 0 ? 2 : 1;  // faces per thread
    constexpr int CH = CN / NH;
    const double gR = gas_gR(p.g);
    for (int i = tid; i < CH * L; i += NT) {
        int itn, il;
        if (DIR == 2) { itn = i % CN; il = i / CN; }
        else { il = i % L; itn = NH * (i / L); }
        int ia, ib;
        LN::coords(il, ia, ib);
        const int ca = wrapi(a0 + ia, nc), cb = wrapi(b0 + ib, nc);
        const int fn = n0 + itn;
        double S[5 + NH][5], Tc[5 + NH];
#pragma unroll
        for (int t = 0; t < 5 + NH; t++) {
            const long idx = cell_index<DIR>(wrapi(fn - 2 + t, nc), ca, cb, nc);
#pragma unroll
            for (int q = 0; q < 5; q++) S[t][q] = W[q * plane + idx];
            if (NH == 2) Tc[t] = temp_gr<double>(S[t], gR);
        }
#pragma unroll
        for (int h = 0; h < NH; h++) {
            double Wl[5], Wr[5];
            if constexpr (NH == 2) weno5_mixed_t(S + h, Tc + h, p.g, Wl, Wr);
            else weno5_mixed(S, p.g, Wl, Wr);
#pragma unroll
            for (int q = 0; q < 5; q++) {
                sW[sw_at<DIR, CN, L>(q, itn + h, il)] = Wl[q];
                sW[sw_at<DIR, CN, L>(5 + q, itn + h, il)] = Wr[q];
            }
        }
    }
}

// The FP64 sweep keeps the cells its chunk's stencils read in LDS: a ring of
// CN + 5 cells of every line of the pencil, 6 values each (5 conserved variables
// and the temperature).  Walking the line by one chunk loads CN new cells per
// line; they are loaded into registers before the flux of the chunk before and
// stored in the ring after it, so HBM and L2 latency pass behind the flux.
// (Reading each stencil from the state array took 30 loads and 6 temperatures
// per face and line where this takes 5 and 1, and the 256^3 sweeps a fifth longer.)
template <int CN>
constexpr int kRing = CN + 5;
template <int DIR, int CN, int L>
__device__ __forceinline__ int ring_at(int v, int slot, int l)
{
    return DIR == 2 ? (v * L + l) * kRing<CN> + slot : (v * kRing<CN> + slot) * L + l;
}
template <int DIR, int CN, int L>
__host__ __device__ constexpr int ring_at_stride()  // doubles between the variables of a cell
{
    return kRing<CN> * L;
}
// ring slot of window position j (cells n0 - 2 + j of the chunk at n0), head h
template <int CN>
__device__ __forceinline__ int ring_slot(int h, int j)
{
    const int k = h + j;
    return k >= kRing<CN> ? k - kRing<CN> : k;
}

// Flux inputs of one side of a face for gks_flux_pair, in the lane's frame, all
// from LDS: the cell from the ring, WENO states and their tangential
// differences from sW.
template <int DIR, int CN, int L>
struct PairIn {
    const double* s;         // the side's slot 0 at the lane's face, line 0
    const double* c;         // ring: variable 0 of the side's cell
    int side;
    int lc, m0, p0, m1, p1;  // own line; lines before and after along the first / second direction
    double two_idx, half_idx;
    static constexpr int kVar = ring_at_stride<DIR, CN, L>();
    __device__ __forceinline__ double at(int q, int line) const
    {
        return s[DIR == 2 ? (q * L + line) * CN : q * (CN * L) + line];
    }
    __device__ __forceinline__ double S(int q) const { return at(q, lc); }
    __device__ __forceinline__ double C(int q) const
    {
        constexpr int n = pair_var<DIR>(0, 1);
        if (q == 1) return side ? -c[n * kVar] : c[n * kVar];
        if (q == 2 || q == 3) return c[(side ? pair_var<DIR>(1, q) : pair_var<DIR>(0, q)) * kVar];
        return c[q * kVar];
    }
    __device__ __forceinline__ double N(int q) const { return (at(q, lc) - C(q)) * two_idx; }
    __device__ __forceinline__ double T(int k, int q) const
    {
        return (k == 0 ? at(q, p0) - at(q, m0) : at(q, p1) - at(q, m1)) * half_idx;
    }
};

// The FP64 sweep: a workgroup of 256 threads walks a pencil of CA x CB lines in
// chunks of CN faces, CN CA CB = 128, two threads per face (gks_flux_pair).
// Otherwise as sweep_body below.
// FACES = true: the fluxes of the faces i+1/2 of cells i go to p.dW (5 planes)
// instead of the flux differences, and there is no lead-in chunk (step_update
// forms the differences of all three directions).
template <int DIR, int V, bool EXT = false, bool GEN = true, bool FACES = false>
__device__ __forceinline__ void sweep_body_pair(const SweepArgs& p, int bid, int nblk, bool remap, double* lds = nullptr)
{
    constexpr int CN = Tile<DIR, V, false>::CN, CA = Tile<DIR, V, false>::CA, CB = Tile<DIR, V, false>::CB;
    constexpr int NT = 256, NL = CA * CB, NF = CN * NL, RC = kRing<CN>;
    using LN = Lines<CA, CB>;
    constexpr int L = LN::L;
    static_assert(2 * NF == NT && CN * L <= NT, "two threads per face, one line cell per thread");
    double* sC;  // cells: the ring
    if constexpr (EXT) {
        sC = lds;
    } else {
        __shared__ double own[sweep_lds_doubles<DIR, V, false>()];
        sC = own;
    }
    double* const sW = sC + 6 * RC * L;   // WENO states of the two sides (5 each), in their lanes' frames
    double* const sF = sW + 10 * CN * L;  // face fluxes of this chunk and the one before

    const int nc = p.nc;
    const long plane = p.plane;
    const double* __restrict__ W = p.W;
    int a0, b0, s;
    sweep_pencil<DIR, CA, CB, GEN, FACES>(p, bid, nblk, remap, a0, b0, s);

    const int tid = threadIdx.x;
    const double dt = *p.dt;
    const double dx = p.dx;
    const int nchunk = p.seg / CN;
    const int seg0 = FACES && s * p.seg > nc - p.seg ? nc - p.seg : s * p.seg;
    const int seg_end = seg0 + p.seg < nc ? seg0 + p.seg : nc;

    // the thread's line and cell (loads, WENO)
    const bool has = tid < CN * L;
    const int il = DIR == 2 ? tid / CN : tid % L, itn = DIR == 2 ? tid % CN : tid / L;
    int lca, lcb;
    {
        int ia, ib;
        LN::coords(has ? il : 0, ia, ib);
        lca = wrapi(a0 + ia, nc);
        lcb = wrapi(b0 + ib, nc);
    }
    auto store = [&](int slot, const double c[5]) {
        double* r = sC + ring_at<DIR, CN, L>(0, slot, il);
        constexpr int st = ring_at_stride<DIR, CN, L>();
#pragma unroll
        for (int q = 0; q < 5; q++) r[q * st] = c[q];
        r[5 * st] = temp_gr<double>(c, gas_gR(p.g));
    };
    // window of the first chunk (the lead-in): cells n - 2 ... n + CN + 2
    constexpr int c0 = FACES ? 0 : -1;
    for (int j = itn; has && j < RC; j += CN) {
        const long idx = cell_index<DIR>(wrapi(seg0 + c0 * CN - 2 + j, nc), lca, lcb, nc);
        double c[5];
#pragma unroll
        for (int q = 0; q < 5; q++) c[q] = W[q * plane + idx];
        store(j, c);
    }
    __syncthreads();

    // the thread's face and side (flux): neighbouring lanes are the two sides of a face
    const int side = tid & 1;
    int tn, ta, tb;
    sweep_face<DIR, CN, CA, CB>(tid >> 1, tn, ta, tb);
    // the thread's cell in the update: the first half of the workgroup takes
    // rho, rho u and rho v, the second rho w and rho E
    int un, ua, ub;
    sweep_face<DIR, CN, CA, CB>(tid & (NF - 1), un, ua, ub);
    const int uc = ua * CB + ub;
    const int q0 = tid < NF ? 0 : 3;

    int h = 0;  // ring slot of cell n0 - 2
    for (int c = c0; c < nchunk; ++c) {
        const int n0 = seg0 + c * CN;  // first face of the chunk (may be < 0 for the lead-in)

        // ---- WENO states of every (face, line) of the chunk, one variable at a
        // time: its six cells are dead before the next one's
        if (has) {
            const double* r[6];
#pragma unroll
            for (int t = 0; t < 6; t++) r[t] = sC + ring_at<DIR, CN, L>(0, ring_slot<CN>(h, itn + t), il);
            constexpr int st = ring_at_stride<DIR, CN, L>();
            double* const o = sW + sw_at<DIR, CN, L>(0, itn, il);
            constexpr int so = L * CN;
            double den[2], m2[2];
#pragma unroll
            for (int q = 0; q < 5; q++) {
                const int v = (q == 4 ? 5 : q) * st;
                double x[2];
                weno_pair(r[0][v], r[1][v], r[2][v], r[3][v], r[4][v], r[5][v], p.g.eps, x[0], x[1]);
#pragma unroll
                for (int d = 0; d < 2; d++) {
                    if (q == 0) den[d] = x[d];
                    else if (q < 4) m2[d] = q == 1 ? x[d] * x[d] : fma(x[d], x[d], m2[d]);
                    else x[d] = fma(den[d] * gas_Rg(p.g), x[d], (0.5 * m2[d]) * g_rcp(den[d]));
                    const int k = pair_slot<DIR>(d, q);
                    o[(5 * d + k) * so] = d && k == 1 ? -x[d] : x[d];
                }
            }
        }
        __syncthreads();

        // ---- loads whose latency the flux hides: the next chunk's new cells, and
        // the sum so far of this chunk's cells
        double cell[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (has && c + 1 < nchunk) {
            const long idx = cell_index<DIR>(wrapi(n0 + CN + 3 + itn, nc), lca, lcb, nc);
#pragma unroll
            for (int q = 0; q < 5; q++) cell[q] = W[q * plane + idx];
        }
        const bool live = c >= 0 && (!GEN || (a0 + ua < nc && b0 + ub < nc && n0 + un < seg_end));
        double old[3] = {0.0, 0.0, 0.0}, was[3] = {0.0, 0.0, 0.0};
        if (!FACES && DIR != 0 && live && p.mode != 0) {
            const long idx = cell_index<DIR>(n0 + un, a0 + ua, b0 + ub, nc);
#pragma unroll
            for (int k = 0; k < 3; k++)
                if (q0 + k < 5) old[k] = p.dW[(q0 + k) * plane + idx];
        }
        if (!FACES && DIR == 2) {
            // the cells themselves: after the flux their ring slots may be rewritten
            const double* const w = sC + ring_at<DIR, CN, L>(0, ring_slot<CN>(h, un + 2), uc);
#pragma unroll
            for (int k = 0; k < 3; k++)
                if (q0 + k < 5) was[k] = w[(q0 + k) * ring_at_stride<DIR, CN, L>()];
        }
        __builtin_amdgcn_sched_barrier(0);

        {
            PairIn<DIR, CN, L> in;
            in.s = sW + sw_at<DIR, CN, L>(5 * side, tn, 0);
            in.lc = ta * CB + tb;
            in.c = sC + ring_at<DIR, CN, L>(0, ring_slot<CN>(h, tn + 2 + side), in.lc);
            in.side = side;
            const int am = LN::id(ta - 1, tb), ap = LN::id(ta + 1, tb);
            const int bm = LN::id(ta, tb - 1), bp = LN::id(ta, tb + 1);
            in.m0 = side ? bm : am;
            in.p0 = side ? bp : ap;
            in.m1 = side ? am : bm;
            in.p1 = side ? ap : bp;
            in.two_idx = p.two_idx;
            in.half_idx = p.half_idx;
            // the collision time is the left cell's
            const double* left = sC + ring_at<DIR, CN, L>(0, ring_slot<CN>(h, tn + 2), in.lc);
            constexpr int st = ring_at_stride<DIR, CN, L>();
            const double tau = collision_time_t(left[0], left[5 * st], p.g);
            double F[5];
            gks_flux_pair(in, tau, dt, dx, p.g, PairSwap{}, F);
            if (side == 0) {
                double* const f = sF + ((c & 1) * 5) * NF + pf_at<DIR, CN, NL>(tn, in.lc);
#pragma unroll
                for (int q = 0; q < 5; q++) f[pair_var<DIR>(0, q) * NF] = F[q];
            }
        }
        __syncthreads();

        // ---- flux differences of the chunk's cells
        if (live) {
            const long idx = cell_index<DIR>(n0 + un, a0 + ua, b0 + ub, nc);
            const double* const f1 = sF + ((c & 1) * 5) * NF + pf_at<DIR, CN, NL>(un, uc);
            const double* const f0 = un ? sF + ((c & 1) * 5) * NF + pf_at<DIR, CN, NL>(un - 1, uc)
                                        : sF + ((~c & 1) * 5) * NF + pf_at<DIR, CN, NL>(CN - 1, uc);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const int q = q0 + k;
                if (q >= 5) break;
                const long o = q * plane + idx;
                if (FACES) {
                    p.dW[o] = f1[q * NF];
                    continue;
                }
                const double dF = f1[q * NF] - f0[q * NF];
                if (DIR == 0 || p.mode == 0) p.dW[o] = dF;
                else if (DIR == 1) p.dW[o] = old[k] + dF;
                else p.Wout[o] = was[k] - p.inv_dx * (old[k] + dF);
            }
        }
        // the new cells take the places of the oldest, which this chunk's WENO and its
        // flux (window positions 2 to CN + 2) have read: the barrier after the flux
        // stands between
        if (has && c + 1 < nchunk) store(ring_slot<CN>(h, itn), cell);
        h = ring_slot<CN>(h, CN);
        __syncthreads();
    }
}

// MIX = true: WENO in FP32 on FP64 stencil differences and the flux with FP32
// slope terms (gks_flux_tf<double, float>), below.  MIX = false: the FP64 path,
// sweep_body_pair.  Two waves per SIMD are requested: the register budget is
// then 256 per lane.  With one wave per SIMD the compiler (ROCm 7.2, gfx950)
// spilled into AGPRs and the x and y instances produced wrong flux differences
// on the GPU (the z instance and every instance built this way match the FP64
// oracle to 1e-14).
//
// sweep_body is the work of one workgroup: block `bid` of the `nblk` blocks of
// one grid (member).  remap = true applies the XCD-aware order to bid.
// EXT = false: the body's own LDS arrays; EXT = true: the caller's buffer lds
// of at least sweep_lds_doubles<DIR, V, true>() doubles (a kernel running several
// bodies shares one buffer between them).
// GEN = true: any grid (tiles and segments may reach past nc); GEN = false:
// only for grids the tile and the segment divide (no line or face of the
// workgroup lies past the grid, so none is masked or wrapped into range: the
// general form's extra live values made the mixed x and y sweeps spill).
// CMP (the z sweep's update): -1 compensated when p.cmp_out is set, 0 plain,
// 1 compensated (the fixed forms leave the other update out of the kernel).
// FACES as in sweep_body_pair.
template <int DIR, bool MIX, int V, bool EXT = false, bool GEN = true, int CMP = -1, bool FACES = false>
__device__ __forceinline__ void sweep_body(const SweepArgs& p, int bid, int nblk, bool remap, double* lds = nullptr)
{
    if constexpr (!MIX) {
        sweep_body_pair<DIR, V, EXT, GEN, FACES>(p, bid, nblk, remap, lds);
        return;
    } else {
    constexpr int CN = Tile<DIR, V, true>::CN, CA = Tile<DIR, V, true>::CA, CB = Tile<DIR, V, true>::CB;
    constexpr int NT = CN * CA * CB;
    static_assert(NT == 256, "every tile variant runs 256 threads, one face each");
    using LN = Lines<CA, CB>;
    constexpr int L = LN::L;
    double* sW;  // WENO states: Wl (0..4), Wr (5..9)
    double* sF;  // face fluxes; slot 0 = face before the chunk
    if constexpr (EXT) {
        sW = lds;
    } else {
        __shared__ double own[sweep_lds_doubles<DIR, V, true>()];
        sW = own;
    }
    sF = sW + 10 * CN * L;

    const int nc = p.nc;
    const long plane = p.plane;
    const double* __restrict__ W = p.W;

    int a0, b0, s;
    sweep_pencil<DIR, CA, CB, GEN, FACES>(p, bid, nblk, remap, a0, b0, s);

    const int tid = threadIdx.x;
    int tn, ta, tb;
    sweep_face<DIR, CN, CA, CB>(tid, tn, ta, tb);
    const int lc = ta * CB + tb;
    // a grid that is not a multiple of the tile: lines past nc (their cells
    // wrap) and faces past the segment's end are computed, not written
    const bool live = !GEN || (a0 + ta < nc && b0 + tb < nc);

    const double dt = *p.dt;
    const double dx = p.dx;
    const int nchunk = p.seg / CN;
    const int seg0 = FACES && s * p.seg > nc - p.seg ? nc - p.seg : s * p.seg;
    const int seg_end = seg0 + p.seg < nc ? seg0 + p.seg : nc;

    SweepIn<DIR, CN, L> in;
    in.W = W;
    in.plane = plane;
    in.s = sW;
    in.tn = tn;
    in.lc = lc;
    in.l_am = LN::id(ta - 1, tb);
    in.l_ap = LN::id(ta + 1, tb);
    in.l_bm = LN::id(ta, tb - 1);
    in.l_bp = LN::id(ta, tb + 1);
    in.two_idx = p.two_idx;
    in.half_idx = p.half_idx;

    for (int c = FACES ? 0 : -1; c < nchunk; ++c) {
        const int n0 = seg0 + c * CN;  // first face of the chunk (may be < 0 for the lead-in)

        weno_chunk<DIR, CN, CA, CB, NT>(p, n0, a0, b0, tid, sW);
        __syncthreads();

        // y sweep: the sum so far of the chunk's cells, loaded ahead of the flux,
        // which hides the latency (256^3, 2 x 8 x 16 tile: 2.16 -> 1.98 ms; the z
        // sweep with its carry has no registers left for it, 2.42 -> 2.58 ms, nor
        // has the persistent step's kernel, 5.56 -> 5.71 ms for 64 members).  Faces
        // alone have no sum (mode 0), but are scheduled better with the branch in
        // than without it (128^3 mixed, 769 against 782 us a step)
        constexpr bool AHEAD = DIR == 1 && (!EXT || FACES);
        const bool upd = c >= 0 && live && (!GEN || n0 + tn < seg_end);
        double old[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (AHEAD && upd && p.mode != 0) {
            const long idx = cell_index<DIR>(n0 + tn, a0 + ta, b0 + tb, nc);
#pragma unroll
            for (int q = 0; q < 5; q++) old[q] = p.dW[q * plane + idx];
            __builtin_amdgcn_sched_barrier(0);
        }
        // ---- one GKS flux per thread
        {
            const int fn = n0 + tn;
            const int ca = GEN ? wrapi(a0 + ta, nc) : a0 + ta, cb = GEN ? wrapi(b0 + tb, nc) : b0 + tb;
            in.iL = cell_index<DIR>(wrapi(fn, nc), ca, cb, nc);
            in.iR = cell_index<DIR>(wrapi(fn + 1, nc), ca, cb, nc);
            double tau;
            {
                double WL[5];
#pragma unroll
                for (int q = 0; q < 5; q++) WL[q] = W[q * plane + in.iL];
                tau = collision_time<double>(WL, p.g);  // symmetric in the momentum slots
            }
            double F[5];
            gks_flux_tf<double, float>(in, tau, dt, dx, p.g, F);
            if constexpr (FACES) {
                if (upd) {
                    const long idx = cell_index<DIR>(n0 + tn, a0 + ta, b0 + tb, nc);
#pragma unroll
                    for (int q = 0; q < 5; q++) p.dW[in.phys(q) * plane + idx] = F[q];
                }
                __syncthreads();  // the next chunk's WENO rewrites sW
                continue;
            }
#pragma unroll
            for (int q = 0; q < 5; q++) sF[sf_at<DIR, CN, CA * CB>(in.phys(q), tn + 1, lc)] = F[q];
        }
        __syncthreads();

        // ---- flux differences of the chunk's cells
        if (upd) {
            const long idx = cell_index<DIR>(n0 + tn, a0 + ta, b0 + tb, nc);
#pragma unroll
            for (int q = 0; q < 5; q++) {
                const double dF = sF[sf_at<DIR, CN, CA * CB>(q, tn + 1, lc)] - sF[sf_at<DIR, CN, CA * CB>(q, tn, lc)];
                const long o = q * plane + idx;
                // the x sweep only ever starts the sum; the y sweep adds to it
                // unless asked for its flux differences alone (mode 0), the z
                // sweep updates unless asked for its flux differences alone
                if (DIR == 0 || p.mode == 0) p.dW[o] = dF;
                else if (DIR == 1) p.dW[o] = (AHEAD ? old[q] : p.dW[o]) + dF;
                else if (CMP == 1 || (CMP < 0 && p.cmp_out)) {
                    // W^{n+1} + e = W^n + (increment + carried error), exactly (TwoSum);
                    // z sweep: n = z, a = x, b = y
                    const long co = q * carry_plane(nc) + carry_index(b0 + tb, a0 + ta, n0 + tn, nc);
                    const double w = W[o];
                    const double y = (double)p.cmp_in[co] - p.inv_dx * (p.dW[o] + dF);
                    const double t = w + y;
                    const double yv = t - w;
                    const double e = (w - (t - yv)) + (y - yv);
                    p.Wout[o] = t;
                    p.cmp_out[co] = (float)e;
                } else {
                    p.Wout[o] = W[o] - p.inv_dx * (p.dW[o] + dF);
                }
            }
        }
        __syncthreads();
        if (tn == CN - 1) {
#pragma unroll
            for (int q = 0; q < 5; q++) sF[sf_at<DIR, CN, CA * CB>(q, 0, lc)] = sF[sf_at<DIR, CN, CA * CB>(q, CN, lc)];
        }
        // the next write of sF slots 1..CN happens after the next chunk's first barrier
    }
    }
}

// ---------------------------------------------------------------------------
// CFL reductions: dt = cfl dx / max(|U| + sqrt(gam p / rho)) over all cells
// (timestep, update.cpp:1031-1054).  A non-physical cell (rho <= 0, p <= 0 or
// not finite) records -1 instead of its block maximum.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_max(double v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// |U| + c of one cell into m; bad: the cell is non-physical
__device__ __forceinline__ void cfl_cell(double den, double m1, double m2, double m3, double e, double gam, double& m,
                                         bool& bad)
{
    const double ir = 1.0 / den;
    const double u = m1 * ir, v = m2 * ir, w = m3 * ir;
    const double Vsqr = u * u + v * v + w * w;
    const double P = (den * (gam - 1)) * (e * ir - 0.5 * Vsqr);
    const double val = sqrt(Vsqr) + sqrt(gam * P * ir);
    if (!(den > 0.0) || !(P > 0.0) || !isfinite(val)) bad = true;
    else m = fmax(m, val);
}

// block maximum m (or -1 where a thread saw a bad cell), written by thread 0 to *out
__device__ __forceinline__ void cfl_block(double m, bool bad, double* out)
{
    __shared__ double sm[4];
    __shared__ int sbad;
    if (threadIdx.x == 0) sbad = 0;
    __syncthreads();
    if (bad) sbad = 1;
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double r = fmax(fmax(sm[0], sm[1]), fmax(sm[2], sm[3]));
        *out = sbad ? -1.0 : r;
    }
    __syncthreads();  // sm, sbad are reused by the block's next call
}

// maximum of |U| + c over cells c0, c0 + stride, ... of one state; thread 0
// writes it (or -1) to *out
__device__ __forceinline__ void cfl_cells(const double* __restrict__ W, long plane, double gam, long c0, long stride,
                                          double* out)
{
    double m = 0.0;
    bool bad = false;
    for (long c = c0 + threadIdx.x; c < plane; c += stride)
        cfl_cell(W[c], W[plane + c], W[2 * plane + c], W[3 * plane + c], W[4 * plane + c], gam, m, bad);
    cfl_block(m, bad, out);
}

// block reduction of n partial maxima (-1 = non-physical state seen) -> dt
__device__ __forceinline__ void cfl_reduce(const double* partial, int n, double cfl, double dx, double* dt, double* vmax,
                                           int* bad, double* hist = nullptr)
{
    double m = 0.0;
    int b = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const double v = partial[i];
        if (v < 0.0) b = 1;
        else m = fmax(m, v);
    }
    __shared__ double sm[4];
    __shared__ int sb[4];
    m = wave_max(m);
    // any-reduction of the flag
    unsigned long long ballot = __ballot(b);
    if ((threadIdx.x & 63) == 0) {
        sm[threadIdx.x >> 6] = m;
        sb[threadIdx.x >> 6] = ballot != 0ull;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const double r = fmax(fmax(sm[0], sm[1]), fmax(sm[2], sm[3]));
        const int anyb = sb[0] | sb[1] | sb[2] | sb[3];
        *vmax = r;
        *bad = anyb;
        const double d = (anyb || !(r > 0.0)) ? 0.0 : cfl * dx / r;
        *dt = d;
        if (hist) *hist = d;
    }
    __syncthreads();  // sm, sb are reused by the block's next call
}

}  // namespace gkm
