// lpt_kernels.hip -- natural tricubic B-spline prefilter, particle sampling and
// Heun advection, and flow / particle statistics on gfx950.
//
// Spline semantics (einspline UBspline_3d_d with NATURAL ends as built by
// get_bsplinep, Interpolation.cpp:3-31): nt = nc+6 knots per axis at the
// padded cell centres, N = nt+2 coefficients per axis, interpolation rows
// (c_i + 4 c_{i+1} + c_{i+2})/6 = f_i and f'' = 0 at both ends, i.e.
// c_1 = f_0, c_nt = f_{nt-1}, a [1 4 1] system for the inner coefficients and
// c_0 = 2c_1 - c_2, c_{nt+1} = 2c_nt - c_{nt-1}.  The 3-D coefficients are the
// tensor product: the line solve is applied along z, then x, then y.
#include "lpt_kernels.hpp"
#include "lpt_device.hpp"

#include <initializer_list>
#include <type_traits>

namespace lpt {

void release(State& s)
{
    (void)hipFree(s.pos);
    (void)hipFree(s.U);
    (void)hipFree(s.G);
    for (int b = 0; b < 2; b++)
        for (int q = 0; q < 3; q++) {
            (void)hipFree(s.coef[b][q]);
            s.coef[b][q] = nullptr;
        }
    for (int f = 0; f < 5; f++) (void)hipFree(s.pcoef[f]);
    (void)hipFree((void*)s.pcs);
    (void)hipFree(s.props);
    (void)hipFree(s.pivots);
    (void)hipFree(s.red);
    (void)hipFree(s.tag);
    (void)hipFree(s.tag2);
    (void)hipFree(s.pos2);
    (void)hipFree(s.keys);
    (void)hipFree(s.perm);
    (void)hipFree(s.sort_tmp);
    s = State();
}

// four waves per block, one z line each
template <int K>
__global__ __launch_bounds__(256) void prefilter_z_kernel(ZArgs z)
{
    const long line = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (line >= (long)z.g.nt * z.g.nt) return;  // uniform over the wave
    prefilter_z_line<K>(line, z);
}

// z pass in place over knot values already in the coefficient box (positions
// [0, nt) of every z line with a, b < nt), as the Laplacian splines need
template <int K>
__global__ __launch_bounds__(256) void knots_z_kernel(double* __restrict__ coef, Geom g, const double* __restrict__ piv)
{
    const long line = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int nt = g.nt, lane = threadIdx.x & 63;
    if (line >= (long)nt * nt) return;
    double* row = coef + ((line / nt) * g.N + line % nt) * g.N;
    double f[K];
#pragma unroll
    for (int j = 0; j < K; j++) {
        const int p = 64 * j + lane;
        f[j] = p < nt ? row[p] : 0.0;
    }
    zline_solve<K>(f, nt, piv, row);  // every lane has read its values before the first store
}

// smallest instantiated chunk count holding nt knots (0: too many)
static int z_chunks(int nt)
{
    const int need = (nt + 63) / 64;
    for (int k : {1, 2, 3, 5, 9, kMaxZChunks})
        if (need <= k) return k;
    return 0;
}

template <typename F>
static hipError_t with_chunks(int k, F&& f)
{
    switch (k) {
    case 1: return f(std::integral_constant<int, 1>());
    case 2: return f(std::integral_constant<int, 2>());
    case 3: return f(std::integral_constant<int, 3>());
    case 5: return f(std::integral_constant<int, 5>());
    case 9: return f(std::integral_constant<int, 9>());
    case kMaxZChunks: return f(std::integral_constant<int, kMaxZChunks>());
    default: return hipErrorInvalidValue;
    }
}

// up to three coefficient boxes of one geometry, solved by one launch per axis
struct CoefSet {
    double* c[3];
};

// Workgroups [f bpf, (f + 1) bpf) solve the lines of box f (bpf = workgroups
// per box).  A workgroup is 256 consecutive lines, so its four waves (one per
// SIMD of a CU) read and write each row as one 2 KB run rather than four 512 B
// runs of unrelated workgroups: the passes are bound by how HBM serves runs at
// a stride of N or N^2 coefficients (0.54 -> 0.53 ms per pass and box at 512^3;
// more loads in flight per wave, or one box per launch against three, measured
// the same).  One such workgroup runs on a CU at a time (dynamic LDS the
// kernel does not touch, 96 KB of the CU's 160 KB): fewer rows in flight at
// once are served faster (x / y pass over u, v, w at three waves per SIMD
// 1.62 / 1.54 ms, at two 1.57 / 1.50, at one 1.44 / 1.41).
constexpr unsigned kInplaceLdsCap = 96 * 1024;  // 1 wave per SIMD

__global__ __launch_bounds__(256) void prefilter_inplace_kernel(CoefSet cs, unsigned bpf, Geom g, int axis,
                                                                 const double* __restrict__ piv)
{
    const unsigned f = blockIdx.x / bpf;
    prefilter_inplace_one((long)(blockIdx.x - f * bpf) * blockDim.x + threadIdx.x, cs.c[f], g, axis, piv);
}

static unsigned blocks_for(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// x then y pass over nf (1..3) boxes
static hipError_t prefilter_xy(const CoefSet& cs, int nf, const Geom& g, const double* pivots, hipStream_t s)
{
    const unsigned bx = blocks_for((long)g.nt * g.N, 256), by = blocks_for((long)g.N * g.N, 256);
    hipLaunchKernelGGL(prefilter_inplace_kernel, dim3(bx * nf), dim3(256), kInplaceLdsCap, s, cs, bx, g, 1, pivots);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(prefilter_inplace_kernel, dim3(by * nf), dim3(256), kInplaceLdsCap, s, cs, by, g, 2, pivots);
    return hipGetLastError();
}

static hipError_t prefilter_xy(double* coef, const Geom& g, const double* pivots, hipStream_t s)
{
    return prefilter_xy(CoefSet{{coef, coef, coef}}, 1, g, pivots, s);
}

static hipError_t launch_z(const ZArgs& z, hipStream_t s)
{
    const unsigned blocks = blocks_for((long)z.g.nt * z.g.nt, 4);
    return with_chunks(z_chunks(z.g.nt), [&](auto k) {
        hipLaunchKernelGGL(prefilter_z_kernel<decltype(k)::value>, dim3(blocks), dim3(256), 0, s, z);
        return hipGetLastError();
    });
}

hipError_t launch_prefilter(const double* W, long plane, int q, double gam, const Geom& g, const double* pivots,
                            double* coef, hipStream_t s)
{
    if (q < 0 || q > 4 || g.nt != g.nc + 6 || g.N != g.nt + 2 || !z_chunks(g.nt)) return hipErrorInvalidValue;
    hipError_t e = launch_z(ZArgs{W, plane, q, 1, gam, g, pivots, {coef, nullptr, nullptr}}, s);
    if (e != hipSuccess) return e;
    return prefilter_xy(coef, g, pivots, s);
}

hipError_t launch_prefilter_velocity(const double* W, long plane, double gam, const Geom& g, const double* pivots,
                                     double* const coef[3], hipStream_t s)
{
    if (g.nt != g.nc + 6 || g.N != g.nt + 2 || !z_chunks(g.nt)) return hipErrorInvalidValue;
    hipError_t e = launch_z(ZArgs{W, plane, 1, 3, gam, g, pivots, {coef[0], coef[1], coef[2]}}, s);
    if (e != hipSuccess) return e;
    return prefilter_xy(CoefSet{{coef[0], coef[1], coef[2]}}, 3, g, pivots, s);
}

// Laplacian of the spline c at every padded knot (eval_UBspline_3d_d_vgl at the
// cell centres, update.cpp:1218-1229).  At a knot the uniform cubic B-spline
// weights are (1, 4, 1)/6 for the value and (1, -2, 1) delta^-2 for the second
// derivative, so the Laplacian is a 27-point stencil on the coefficients.
// The result lands at the knot positions of the coefficient box `lap`.
// A thread walks `march` knots of a column along the slowest axis and keeps the
// two in-plane sums of three coefficient planes: 9 loads a knot where a knot by
// itself takes 27, and no index divisions inside.  What is left is the box read
// and written once (240^3: 177 -> 93 us,
// 2.5 TB/s; 128^3: 28 -> 18).
__global__ __launch_bounds__(256) void lap_knots_kernel(const double* __restrict__ c, Geom g, int march,
                                                        double* __restrict__ lap)
{
    const int nt = g.nt;
    const unsigned col = blockIdx.x * 256u + threadIdx.x;
    if (col >= (unsigned)nt * (unsigned)nt) return;
    const long N = g.N;
    const int b = (int)(col / (unsigned)nt), k = (int)(col - (unsigned)b * nt);
    const int a0 = blockIdx.y * march, a1 = a0 + march < nt ? a0 + march : nt;
    const double w[3] = {1.0 / 6.0, 4.0 / 6.0, 1.0 / 6.0}, d2[3] = {1.0, -2.0, 1.0};
    const double scale = g.dinv * g.dinv;
    const double* at = c + ((long)a0 * N + b) * N + k;
    // plane sums: V weights (1, 4, 1) both ways, H second differences along x and z
    auto plane = [&](double& V, double& H) {
        V = H = 0.0;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const double* row = at + j * N;
            const double rv = w[0] * row[0] + w[1] * row[1] + w[2] * row[2];
            V += w[j] * rv;
            H += d2[j] * rv + w[j] * (d2[0] * row[0] + d2[1] * row[1] + d2[2] * row[2]);
        }
        at += N * N;
    };
    double V0, V1, V2, H0, H1, H2;
    plane(V0, H0);
    plane(V1, H1);
    double* out = lap + ((long)a0 * N + b) * N + k;
#pragma unroll 2
    for (int a = a0; a < a1; a++, out += N * N) {
        plane(V2, H2);
        *out = ((d2[0] * V0 + d2[1] * V1 + d2[2] * V2) + (w[0] * H0 + w[1] * H1 + w[2] * H2)) * scale;
        V0 = V1;
        V1 = V2;
        H0 = H1;
        H1 = H2;
    }
}

// Cells a thread of the marching kernels walks on a cube of n^3: 16, or as few as
// leave two workgroups per CU, since on small grids the walk is a chain of loads
// with most of the chip idle (32^3: statistics 26.9 us with 16, 10.0 with 1; a cell a
// thread without the walk took 9.5; Laplacian 7.0, 3.0 and 3.1).
static int march_of(int n)
{
    int m = 16;
    while (m > 1 && (long)blocks_for((long)n * n, 256) * blocks_for(n, m) < 512) m /= 2;
    return m;
}

hipError_t launch_lap_spline(const double* c, const Geom& g, const double* pivots, double* lap, hipStream_t s)
{
    if (c == lap || g.nt != g.nc + 6 || g.N != g.nt + 2 || !z_chunks(g.nt)) return hipErrorInvalidValue;
    const int march = march_of(g.nt);
    const dim3 grid(blocks_for((long)g.nt * g.nt, 256), blocks_for(g.nt, march));
    hipLaunchKernelGGL(lap_knots_kernel, grid, dim3(256), 0, s, c, g, march, lap);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    e = with_chunks(z_chunks(g.nt), [&](auto k) {
        hipLaunchKernelGGL(knots_z_kernel<decltype(k)::value>, dim3(blocks_for((long)g.nt * g.nt, 4)), dim3(256), 0, s,
                           lap, g, pivots);
        return hipGetLastError();
    });
    if (e != hipSuccess) return e;
    return prefilter_xy(lap, g, pivots, s);
}

// Block order for the tracer gathers: the hardware deals workgroups
// round-robin over the 8 XCDs, each with its own L2.  Block b runs the tracers
// of block (b mod 8) G/8 + b/8 (G a multiple of 8), so each XCD walks a
// contiguous range of the block-sorted tracers (lpt_sort.hip) and neighbouring
// cell blocks, whose stencils share cache lines, meet in the same L2.  At
// 512^3 with 2^22 tracers the two together bring the bytes fetched past L2 per
// sample / Heun launch from 12.9 / 15.0 GiB to 4.5 / 4.7 GiB (the u, v, w
// coefficients are 3.1 GiB); the remap with the row-major cell sort left them
// at 12.8 / 14.9 GiB.
__device__ __forceinline__ unsigned xcd_block()
{
    const unsigned b = blockIdx.y * gridDim.x + blockIdx.x, nb = gridDim.x * gridDim.y;  // thread_grid
    return (nb & 7) ? b : (b & 7) * (nb >> 3) + (b >> 3);
}

// Resident tracer waves per SIMD for the gathers at 512^3, 2^22 tracers:
// more waves in flight fetch more distinct stencils at once and lose cache
// hits (sample at 64 VGPRs, up to 8 waves: 1.90 ms; capped at 4: 1.81 ms, at
// 3, 5, 6: 1.86, 1.84, 1.87 ms; Heun at 6 waves: 1.48 ms, capped at 3: 1.40
// ms, at 2 and 4: 1.47, 1.45 ms).  The cap is dynamic LDS that the kernels do
// not touch: 160 KB of LDS per CU hold four workgroups of 36 KB or three of
// 48 KB, a workgroup being one wave per SIMD.
constexpr unsigned kSampleLdsCap = 36 * 1024;  // 4 waves per SIMD
constexpr unsigned kHeunLdsCap = 48 * 1024;    // 3 waves per SIMD

__global__ __launch_bounds__(256) void sample_kernel(long np, const double* __restrict__ pos, const double* __restrict__ cu,
                                                     const double* __restrict__ cv, const double* __restrict__ cw, Geom g,
                                                     double* __restrict__ U, double* __restrict__ G)
{
    const long t = (long)xcd_block() * blockDim.x + threadIdx.x;  // four threads per tracer
    if ((t >> 2) < np) sample_quad(t >> 2, (int)(t & 3), pos, cu, cv, cw, g, U, G);
}

hipError_t launch_sample(long np, const double* pos, const double* const cu[3], const Geom& g, double* U, double* G,
                         hipStream_t s)
{
    if (np <= 0) return hipSuccess;
    hipLaunchKernelGGL(sample_kernel, thread_grid(4 * np), dim3(256), kSampleLdsCap, s, np, pos, cu[0], cu[1],
                       cu[2], g, U, G);
    return hipGetLastError();
}

// Particle::getParticleProp (ParticleTrack.cpp:99-113): value + gradient of rho,
// u, v, w and of the three velocity Laplacians, value + gradient + Hessian of p,
// at each particle.  cs = {rho, u, v, w, p, lap u, lap v, lap w} splines.  Row
// tag[p] of out receives the kPropWidth members in the order of the reference's
// Particle (ParticleTrack.h:21-22): DEN, U[3], P, gradD[3], gradU[3], gradV[3],
// gradW[3], gradP[3], lapU, lapV, lapW, hessP[9], gradLapU[3], gradLapV[3],
// gradLapW[3]; vectors over (y, x, z), hessP row-major over (y, x, z).
// A quad of lanes per tracer and field (sample_quad's way of reading a stencil),
// field after field: a thread per tracer left 1-4 waves per SIMD waiting on their
// gathers one field after the other (10^5 tracers at
// 240^3, where they touch most of the eight fields' 950 MB: 347 -> 215 us; 2^18 at
// 128^3: 318 -> 172).
__global__ __launch_bounds__(256) void props_kernel(long np, const double* __restrict__ pos, const int* __restrict__ tag,
                                                    const double* const* __restrict__ cs, Geom g,
                                                    double* __restrict__ out)
{
    const int f = blockIdx.z;
    const long t = thread_at(blockIdx.x, blockIdx.y, threadIdx.x);
    const long p = t >> 2;
    const int lane = (int)(t & 3);
    if (p >= np) return;
    // output slots of value and gradient per field
    const int vslot = f < 5 ? f : f + 15, gslot = f < 5 ? 5 + 3 * f : 17 + 3 * f;
    double* o = out + (long)tag[p] * kPropWidth;
    double r[4], h[9];  // value and gradient (y, x, z), Hessian
    if (g.drop && isnan(pos[3 * p])) {  // dropped tracer: a row of NaN
#pragma unroll
        for (int k = 0; k < 4; k++) r[k] = __builtin_nan("");
#pragma unroll
        for (int k = 0; k < 9; k++) h[k] = __builtin_nan("");
    } else {
        const Loc Ly = locate(pos[3 * p + 0], g, true);
        const Loc Lx = locate(pos[3 * p + 1], g, true);
        const Loc Lz = locate(pos[3 * p + 2], g, true);
        const double wz = pick4(Lz.w, lane), dz = pick4(Lz.d, lane);
        const long N = g.N;
        const double* cf = cs[f] + ((long)Ly.i * N + Lx.i) * N + Lz.i + lane;
        // second-derivative weights of the cubic B-spline
        auto second = [&](double t, double q[4]) {
            const double d2 = g.dinv * g.dinv;
            q[0] = (1 - t) * d2;
            q[1] = (3 * t - 2) * d2;
            q[2] = (1 - 3 * t) * d2;
            q[3] = t * d2;
        };
        // this lane's column of the sums: value, d/dy, d/dx and, for the pressure, the second ones
        double P = 0, Py = 0, Px = 0, Pyy = 0, Pxx = 0, Pyx = 0;
        double hy[4], hx[4];
        if (f == 4) {
            second(Ly.t, hy);
            second(Lx.t, hx);
        }
#pragma unroll
        for (int a = 0; a < 4; a++) {
            double s = 0, sx = 0, sxx = 0;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const double c = cf[((long)a * N + b) * N];
                s += Lx.w[b] * c;
                sx += Lx.d[b] * c;
                if (f == 4) sxx += hx[b] * c;
            }
            P += Ly.w[a] * s;
            Py += Ly.d[a] * s;
            Px += Ly.w[a] * sx;
            if (f == 4) {
                Pyy += hy[a] * s;
                Pxx += Ly.w[a] * sxx;
                Pyx += Ly.d[a] * sx;
            }
        }
        r[0] = quad_sum(wz * P);
        r[1] = quad_sum(wz * Py);
        r[2] = quad_sum(wz * Px);
        r[3] = quad_sum(dz * P);
        if (f == 4) {
            double hz[4];
            second(Lz.t, hz);
            h[0] = quad_sum(wz * Pyy);
            h[1] = h[3] = quad_sum(wz * Pyx);
            h[2] = h[6] = quad_sum(dz * Py);
            h[4] = quad_sum(wz * Pxx);
            h[5] = h[7] = quad_sum(dz * Px);
            h[8] = quad_sum(pick4(hz, lane) * P);
        }
    }
    o[lane == 0 ? vslot : gslot + lane - 1] = pick4(r, lane);
    if (f == 4) {
        o[23 + lane] = pick4(h, lane);
        o[27 + lane] = pick4(h + 4, lane);
        if (lane == 0) o[31] = h[8];
    }
}

hipError_t launch_props(long np, const double* pos, const int* tag, const double* const* cs_dev, const Geom& g,
                        double* out, hipStream_t s)
{
    if (np <= 0) return hipSuccess;
    hipLaunchKernelGGL(props_kernel, thread_grid(4 * np, 8), dim3(256), 0, s, np, pos, tag, cs_dev, g, out);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void heun_kernel(long np, double* __restrict__ pos, const double* __restrict__ U,
                                                   const double* __restrict__ cu, const double* __restrict__ cv,
                                                   const double* __restrict__ cw, Geom g, const double* __restrict__ dtp)
{
    const long t = (long)xcd_block() * blockDim.x + threadIdx.x;  // four threads per tracer
    if ((t >> 2) < np) heun_quad(t >> 2, (int)(t & 3), pos, U, cu, cv, cw, g, *dtp);
}

hipError_t launch_heun(long np, double* pos, const double* U, const double* const cn[3], const Geom& g,
                       const double* dt, hipStream_t s)
{
    if (np <= 0) return hipSuccess;
    hipLaunchKernelGGL(heun_kernel, thread_grid(4 * np), dim3(256), kHeunLdsCap, s, np, pos, U, cn[0], cn[1],
                       cn[2], g, dt);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Ensemble: the prefilter passes, sampling and Heun of every member in one
// launch each.  Block b belongs to the entry e with first[e] <= b < first[e+1]
// (binary search; uniform over the block) and runs the single-context body with
// that entry's arguments and block index b - first[e].
// ---------------------------------------------------------------------------
template <int K>
__global__ __launch_bounds__(256) void ens_prefilter_z_kernel(const ZArgs* __restrict__ zs,
                                                              const int* __restrict__ first, int n)
{
    const int e = ens_entry(first, n, blockIdx.x);
    const ZArgs z = zs[e];
    const long line = (long)(blockIdx.x - first[e]) * 4 + (threadIdx.x >> 6);
    if (line >= (long)z.g.nt * z.g.nt) return;  // uniform over the wave
    prefilter_z_line<K>(line, z);
}

__global__ __launch_bounds__(64) void ens_prefilter_inplace_kernel(const EnsLine* __restrict__ lines,
                                                                   const int* __restrict__ first, int n, int axis)
{
    const int e = ens_entry(first, n, blockIdx.x);
    const EnsLine L = lines[e];
    prefilter_inplace_one((long)(blockIdx.x - first[e]) * 64 + threadIdx.x, L.coef, L.g, axis, L.piv);
}

__global__ __launch_bounds__(256) void ens_sample_kernel(const EnsPart* __restrict__ parts, const int* __restrict__ first,
                                                         int n)
{
    const int e = ens_entry(first, n, blockIdx.x);
    const EnsPart P = parts[e];
    const long t = (long)(blockIdx.x - first[e]) * 256 + threadIdx.x;  // four threads per tracer
    if ((t >> 2) < P.np) sample_quad(t >> 2, (int)(t & 3), P.pos, P.c[0], P.c[1], P.c[2], P.g, P.U, P.G);
}

__global__ __launch_bounds__(256) void ens_heun_kernel(const EnsPart* __restrict__ parts, const int* __restrict__ first,
                                                       int n)
{
    const int e = ens_entry(first, n, blockIdx.x);
    const EnsPart P = parts[e];
    const long t = (long)(blockIdx.x - first[e]) * 256 + threadIdx.x;  // four threads per tracer
    if ((t >> 2) < P.np) heun_quad(t >> 2, (int)(t & 3), P.pos, P.U, P.c[0], P.c[1], P.c[2], P.g, *P.dt);
}

int ens_z_blocks(const Geom& g) { return (int)blocks_for((long)g.nt * g.nt, 4); }

int ens_xy_blocks(const Geom& g, int axis)
{
    return (int)blocks_for(axis == 1 ? (long)g.nt * g.N : (long)g.N * g.N, 64);
}

int ens_z_chunks(int nt_max) { return z_chunks(nt_max); }

int ens_particle_blocks(long np) { return (int)blocks_for(4 * np, 256); }  // four threads per tracer

hipError_t launch_ens_prefilter(const ZArgs* zs, const int* zfirst, int nz, int zblk, int zchunks,
                                const EnsLine* lines, const int* lfirst, int nl, const int lblk[2], hipStream_t s)
{
    if (nz <= 0) return hipSuccess;
    hipError_t e = with_chunks(zchunks, [&](auto k) {
        hipLaunchKernelGGL(ens_prefilter_z_kernel<decltype(k)::value>, dim3(zblk), dim3(256), 0, s, zs, zfirst, nz);
        return hipGetLastError();
    });
    for (int axis = 1; axis <= 2 && e == hipSuccess; axis++) {
        hipLaunchKernelGGL(ens_prefilter_inplace_kernel, dim3(lblk[axis - 1]), dim3(64), 0, s, lines,
                           lfirst + (axis - 1) * (nl + 1), nl, axis);
        e = hipGetLastError();
    }
    return e;
}

hipError_t launch_ens_sample(const EnsPart* parts, const int* first, int n, int nblk, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(ens_sample_kernel, dim3(nblk), dim3(256), 0, s, parts, first, n);
    return hipGetLastError();
}

hipError_t launch_ens_heun(const EnsPart* parts, const int* first, int n, int nblk, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(ens_heun_kernel, dim3(nblk), dim3(256), 0, s, parts, first, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Statistics.  Velocity gradients at cell centres come from the spline at its
// knots, where the uniform cubic B-spline reduces to the 3-point stencils
// (1,4,1)/6 (value) and (-1,0,1)/(2 delta) (derivative) on the coefficients.
// Block partial sums (wave shuffles + LDS) go to red[]; the host adds the
// kStatBlocks partials in a fixed order.
// ---------------------------------------------------------------------------
template <int K>
__device__ __forceinline__ void block_sum(double (&v)[K], double* out)
{
    __shared__ double sm[4][K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        double x = v[k];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
        v[k] = x;
    }
    const int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < K; k++) sm[wv][k] = v[k];
    __syncthreads();
    if (threadIdx.x < K) out[threadIdx.x] = sm[0][threadIdx.x] + sm[1][threadIdx.x] + sm[2][threadIdx.x] + sm[3][threadIdx.x];
}

__global__ __launch_bounds__(256) void stats_kernel(const double* __restrict__ W, long plane, const double* __restrict__ cu,
                                                    const double* __restrict__ cv, const double* __restrict__ cw, Geom g,
                                                    StatParams sp, int march, double* __restrict__ red)
{
    // sums: 0 tke, 1 diss, 2 sijsij, 3 enstrophy, 4-6 d2, 7-9 d3, 10-12 d4, 13 P, 14 T, 15 1/rho
    double acc[16];
#pragma unroll
    for (int k = 0; k < 16; k++) acc[k] = 0.0;
    const int nc = g.nc;
    const long N = g.N;
    const double w0 = 1.0 / 6.0, w1 = 4.0 / 6.0;
    const double d = 0.5 * g.dinv;
    const double* cs[3] = {cu, cv, cw};
    // A block takes 256 columns along y, `march` cells of them at a time, and a
    // thread keeps three planes' in-plane sums of each field: 27 coefficient loads
    // a cell where a cell by itself takes 81.  With two or three waves per SIMD
    // the time was the loads' latency, once for the coefficients and once for the
    // state (240^3: 548 us, marching alone 562); the next cell's loads before this
    // one's arithmetic: 304 us, 128^3 81 -> 47.
    const unsigned cols = (unsigned)nc * (unsigned)nc, cblk = (cols + 255) / 256;
    const unsigned items = cblk * (unsigned)((nc + march - 1) / march);
    for (unsigned it = blockIdx.x; it < items; it += gridDim.x) {
    const unsigned sg = it / cblk, col = (it - sg * cblk) * 256 + threadIdx.x;
    if (col >= cols) continue;
    const int i = (int)(col / (unsigned)nc), k = (int)(col - (unsigned)i * nc);
    const int j0 = (int)sg * march, j1 = j0 + march < nc ? j0 + march : nc;
    // knot (j+3, i+3, k+3): coefficient block starts at (j+3, i+3, k+3) with t = 0
    long at = ((long)(j0 + 3) * N + (i + 3)) * N + (k + 3);
    struct Plane {
        double v, gx, gz;
    } pl[3][3];  // [plane][field]
    double raw[3][9], w[5];
    auto load = [&] {
#pragma unroll
        for (int f = 0; f < 3; f++)
#pragma unroll
            for (int b = 0; b < 9; b++) raw[f][b] = cs[f][at + (b / 3) * N + b % 3];
        at += N * N;
    };
    auto sums = [&](Plane q[3]) {
#pragma unroll
        for (int f = 0; f < 3; f++) {
            double rv[3], rd[3];
#pragma unroll
            for (int b = 0; b < 3; b++) {
                rv[b] = w0 * (raw[f][3 * b] + raw[f][3 * b + 2]) + w1 * raw[f][3 * b + 1];
                rd[b] = d * (raw[f][3 * b + 2] - raw[f][3 * b]);
            }
            q[f].v = w0 * (rv[0] + rv[2]) + w1 * rv[1];
            q[f].gx = d * (rv[2] - rv[0]);
            q[f].gz = w0 * (rd[0] + rd[2]) + w1 * rd[1];
        }
    };
    auto cell = [&](int j) {
#pragma unroll
        for (int q = 0; q < 5; q++) w[q] = W[q * plane + (long)j * cols + col];
    };
    load();
    sums(pl[0]);
    load();
    sums(pl[1]);
    load();
    cell(j0);
    for (int j = j0; j < j1; j++) {
        sums(pl[2]);
        const double den = w[0], m1 = w[1], m2 = w[2], m3 = w[3], en = w[4];
        // the next cell's loads pass behind this one's arithmetic (one plane past
        // the last cell's is still in the box)
        load();
        cell(j + 1 < j1 ? j + 1 : j);
        __builtin_amdgcn_sched_barrier(0);
        double val[3], gr[3][3];  // gr[f] = d/dy, d/dx, d/dz
#pragma unroll
        for (int f = 0; f < 3; f++) {
            val[f] = w0 * (pl[0][f].v + pl[2][f].v) + w1 * pl[1][f].v;
            gr[f][0] = d * (pl[2][f].v - pl[0][f].v);
            gr[f][1] = w0 * (pl[0][f].gx + pl[2][f].gx) + w1 * pl[1][f].gx;
            gr[f][2] = w0 * (pl[0][f].gz + pl[2][f].gz) + w1 * pl[1][f].gz;
            pl[0][f] = pl[1][f];
            pl[1][f] = pl[2][f];
        }
        const double ir = 1.0 / den;
        const double uu = m1 * ir, vv = m2 * ir, ww = m3 * ir;
        const double Vsqr = uu * uu + vv * vv + ww * ww;
        const double P = (den * (sp.gam - 1)) * (en * ir - 0.5 * Vsqr);
        const double T = P / (sp.R * den);
        const double dudx = gr[0][1], dudy = gr[0][0], dudz = gr[0][2];
        const double dvdx = gr[1][1], dvdy = gr[1][0], dvdz = gr[1][2];
        const double dwdx = gr[2][1], dwdy = gr[2][0], dwdz = gr[2][2];
        const double x = T / sp.T0;
        const double mu = sp.mu0 * (x * sqrt(x)) * (sp.T0 + 110.4) / (T + 110.4);
        acc[0] += den * (val[0] * val[0] + val[1] * val[1] + val[2] * val[2]);
        acc[1] += mu * (dudx * dudx + dudy * dudy + dudz * dudz + dvdx * dvdx + dvdy * dvdy + dvdz * dvdz +
                        dwdx * dwdx + dwdy * dwdy + dwdz * dwdz);
        const double s1 = dudy + dvdx, s2 = dudz + dwdx, s3 = dwdy + dvdz;
        acc[2] += dudx * dudx + 0.5 * s1 * s1 + 0.5 * s2 * s2 + 0.5 * s3 * s3 + dvdy * dvdy + dwdz * dwdz;
        const double o1 = dwdy - dvdz, o2 = dudz - dwdx, o3 = dvdx - dudy;
        acc[3] += o1 * o1 + o2 * o2 + o3 * o3;
        const double dd[3] = {dudx, dvdy, dwdz};
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const double s = dd[a] * dd[a];
            acc[4 + a] += s;
            acc[7 + a] += s * dd[a];
            acc[10 + a] += s * s;
        }
        acc[13] += P;
        acc[14] += T;
        acc[15] += ir;
    }
    }
    block_sum<16>(acc, red + 32 * blockIdx.x);
}

__global__ __launch_bounds__(256) void stats2_kernel(const double* __restrict__ W, long plane, StatParams sp, double pm,
                                                     double tm, double vm, double* __restrict__ red)
{
    double acc[3] = {0, 0, 0};
    for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < plane; c += (long)gridDim.x * blockDim.x) {
        const double den = W[c], ir = 1.0 / den;
        const double uu = W[plane + c] * ir, vv = W[2 * plane + c] * ir, ww = W[3 * plane + c] * ir;
        const double P = (den * (sp.gam - 1)) * (W[4 * plane + c] * ir - 0.5 * (uu * uu + vv * vv + ww * ww));
        const double T = P / (sp.R * den);
        acc[0] += (pm - P) * (pm - P);
        acc[1] += (tm - T) * (tm - T);
        acc[2] += (vm - ir) * (vm - ir);
    }
    block_sum<3>(acc, red + 32 * blockIdx.x + 16);
}

hipError_t launch_stats(const double* W, long plane, const double* const cu[3], const Geom& g, const StatParams& sp,
                        double* red, hipStream_t s)
{
    hipLaunchKernelGGL(stats_kernel, dim3(kStatBlocks), dim3(256), 0, s, W, plane, cu[0], cu[1], cu[2], g, sp,
                       march_of(g.nc), red);
    return hipGetLastError();
}

hipError_t launch_stats2(const double* W, long plane, const StatParams& sp, double pm, double tm, double vm,
                         double* red, hipStream_t s)
{
    hipLaunchKernelGGL(stats2_kernel, dim3(kStatBlocks), dim3(256), 0, s, W, plane, sp, pm, tm, vm, red);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void pstats_kernel(long np, const double* __restrict__ U, const double* __restrict__ G,
                                                     double* __restrict__ red)
{
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (long p = (long)blockIdx.x * blockDim.x + threadIdx.x; p < np; p += (long)gridDim.x * blockDim.x) {
        const double* u = U + 3 * p;
        const double* gg = G + 9 * p;
        acc[0] += u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
        const double dudy = gg[0], dudx = gg[1], dudz = gg[2];
        const double dvdy = gg[3], dvdx = gg[4], dvdz = gg[5];
        const double dwdy = gg[6], dwdx = gg[7], dwdz = gg[8];
        const double s1 = dudy + dvdx, s2 = dudz + dwdx, s3 = dwdy + dvdz;
        acc[1] += dudx * dudx + 0.5 * s1 * s1 + 0.5 * s2 * s2 + 0.5 * s3 * s3 + dvdy * dvdy + dwdz * dwdz;
        acc[2] += dudx * dudx;
        acc[3] += dudx * dudx * dudx;
        acc[4] += dwdz * dwdz;
        acc[5] += dwdz * dwdz * dwdz;
    }
    block_sum<6>(acc, red + 8 * blockIdx.x);
}

hipError_t launch_pstats(long np, const double* U, const double* G, double* red, hipStream_t s)
{
    hipLaunchKernelGGL(pstats_kernel, dim3(kStatBlocks), dim3(256), 0, s, np, U, G, red);
    return hipGetLastError();
}

}  // namespace lpt
