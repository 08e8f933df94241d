// gkm_kernels.hip -- gfx950 kernels of the GKM-WENO Eulerian step.
//
// One fused kernel per sweep direction replaces the reference's derivs*_Kernel,
// flip_Kernel, flux, flipBack_Kernel and update_Kernel chain
// (GPUupdate.cu:119-202): WENO states of every face a workgroup needs are
// built once into LDS, each thread (mixed precision) or pair of threads (FP64)
// then evaluates one GKS face flux, and the flux differences are formed in LDS
// and accumulated per cell.  Interface states never leave LDS, nor do the
// fluxes of the sweeps.  Small grids step in two launches instead (below), whose
// 15 planes of fluxes go through memory.
#include "gkm_kernels.hpp"
#include "gkm_pair.hpp"
#include "gkm_sweep.hpp"

namespace gkm {

template <int DIR, bool MIX, int V, bool GEN, int CMP>
__global__ __launch_bounds__(256, 2) void sweep_kernel(SweepArgs p)
{
    sweep_body<DIR, MIX, V, false, GEN, CMP>(p, blockIdx.x, gridDim.x, true);
}

// the entry a block belongs to: first[k] <= g < first[k + 1], 0 <= k < n
__device__ __forceinline__ int entry_of(const int* __restrict__ first, int n, int g)
{
    int lo = 0, hi = n;  // first[lo] <= g < first[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (first[mid] <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

// One launch for the sweeps of every member of an ensemble: member m owns the
// blocks [first[m], first[m+1]) of the grid, in launch order.  Unlike the
// single-grid sweep there is no XCD-grouped reorder: members' workgroups
// differ in length (a 64^3 pencil has twice the chunks of a 32^3 one), and
// contiguous ranges per XCD would hand one XCD the long ones; dealt round-robin,
// every XCD gets the same mix (64 members at 32^3-64^3: 5.34 against 5.90 ms
// per step).
template <int DIR, bool MIX, int V, bool GEN, int CMP>
__global__ __launch_bounds__(256, 2) void ens_sweep_kernel(const SweepArgs* __restrict__ members,
                                                          const int* __restrict__ first, int nmem)
{
    const int m = entry_of(first, nmem, blockIdx.x);
    const SweepArgs p = members[m];
    sweep_body<DIR, MIX, V, false, GEN, CMP>(p, blockIdx.x - first[m], first[m + 1] - first[m], false);
}

static int cdiv(int a, int b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------------------
// Step of a small grid in two launches.  A 32^3 sweep is 256 workgroups of two
// chunks, one of them the lead-in: three sweeps in turn leave half the chip idle,
// do every face twice and pay three launches.  Here one launch computes the face
// fluxes of all three directions (independent of each other) with no lead-in,
// and a second one the update (the sweeps' expressions in their order: equal to
// them bit for bit) and, in a free-running loop, the CFL maximum of the new
// state; its last workgroup forms the next dt.  On a grid that no tile divides
// the last pencils and segments move back into the grid, where the sweeps' reach
// past it and mask (100^3 mixed, us per step: 647 -> 418).
// ---------------------------------------------------------------------------
struct FaceArgs {
    SweepArgs dir[3];
    int first[4];  // blocks [first[d], first[d+1]) sweep direction d
};
template <bool MIX>
__global__ __launch_bounds__(256, 2) void faces_kernel(FaceArgs a)
{
    __shared__ double lds[max3(sweep_lds_doubles<0, 0, MIX>(), sweep_lds_doubles<1, 0, MIX>(), sweep_lds_doubles<2, 0, MIX>())];
    const int b = blockIdx.x;
    if (b < a.first[1]) sweep_body<0, MIX, 0, true, false, 0, true>(a.dir[0], b, a.first[1], true, lds);
    else if (b < a.first[2]) sweep_body<1, MIX, 0, true, false, 0, true>(a.dir[1], b - a.first[1], a.first[2] - a.first[1], true, lds);
    else sweep_body<2, MIX, 0, true, false, 0, true>(a.dir[2], b - a.first[2], a.first[3] - a.first[2], true, lds);
}

// cell c of the next state, into t and memory
template <bool CMP>
__device__ __forceinline__ void update_cell(const UpdateArgs& a, long c, double t[5])
{
    const int nc = a.nc;
    // plane < 2^31 (small_step_ok); a 64-bit division is some 100 instructions
    const unsigned row = (unsigned)c / (unsigned)nc;
    const int z = (int)((unsigned)c - row * nc), y = (int)(row / (unsigned)nc), x = (int)(row - (unsigned)y * nc);
    const long cx = x ? c - nc : c + (long)(nc - 1) * nc;
    const long cy = y ? c - (long)nc * nc : c + (long)(nc - 1) * nc * nc;
    const long cz = z ? c - 1 : c + nc - 1;
#pragma unroll
    for (int q = 0; q < 5; q++) {
        const double *Fx = a.F + q * a.plane, *Fy = Fx + 5 * a.plane, *Fz = Fy + 5 * a.plane;
        const double dW = (Fx[c] - Fx[cx]) + (Fy[c] - Fy[cy]);
        const double dF = Fz[c] - Fz[cz];
        if constexpr (CMP) {  // TwoSum, as in sweep_body
            const long co = q * carry_plane(nc) + carry_index(y, x, z, nc);
            const double w = a.W[q * a.plane + c];
            const double d = (double)a.cmp_in[co] - a.inv_dx * (dW + dF);
            t[q] = w + d;
            const double dv = t[q] - w;
            a.cmp_out[co] = (float)((w - (t[q] - dv)) + (d - dv));
        } else {
            t[q] = a.W[q * a.plane + c] - a.inv_dx * (dW + dF);
        }
        a.Wout[q * a.plane + c] = t[q];
    }
}

template <bool CMP>
__global__ __launch_bounds__(256) void step_update_kernel(UpdateArgs a)
{
    double m = 0.0;
    bool bad = false;
    for (long c = (long)blockIdx.x * 256 + threadIdx.x; c < a.plane; c += (long)gridDim.x * 256) {
        double t[5];
        update_cell<CMP>(a, c, t);
        if (a.partial) cfl_cell(t[0], t[1], t[2], t[3], t[4], a.gam, m, bad);
    }
    if (!a.partial) return;
    __shared__ int last;
    __shared__ double mine;
    cfl_block(m, bad, &mine);
    if (threadIdx.x == 0) {
        // the block's maximum is written through to where every XCD sees it, and
        // there before the ticket: a release fence would write the whole L2 back,
        // once per block (64^3: 30 us a step)
        __hip_atomic_store(a.partial + blockIdx.x, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const int k = __hip_atomic_fetch_add(a.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = k == (int)gridDim.x - 1;
        if (last) __hip_atomic_store(a.ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
    }
    __syncthreads();
    if (!last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    cfl_reduce(a.partial, gridDim.x, a.cfl, a.dx, a.dt, a.vmax, a.bad, a.hist);
}

// The same two launches for every member of an ensemble: entry d n + m of
// members is member m's faces of direction d, with the blocks [first[k],
// first[k + 1]).  Against the three ens_sweep launches every lead-in chunk and
// two of the launches' ends are gone (8 x 32^3, 8 x 48^3 and 4 x 64^3 mixed with
// 8192 tracers each, us a step: sweeps 1009 -> faces 745 + update 96, all 1264 ->
// 1095).
template <bool MIX>
__global__ __launch_bounds__(256, 2) void ens_faces_kernel(const SweepArgs* __restrict__ members,
                                                          const int* __restrict__ first, int nmem)
{
    __shared__ double lds[max3(sweep_lds_doubles<0, 0, MIX>(), sweep_lds_doubles<1, 0, MIX>(), sweep_lds_doubles<2, 0, MIX>())];
    const int k = entry_of(first, 3 * nmem, blockIdx.x);
    const SweepArgs p = members[k];
    const int b = blockIdx.x - first[k], nblk = first[k + 1] - first[k];
    if (k < nmem) sweep_body<0, MIX, 0, true, false, 0, true>(p, b, nblk, false, lds);
    else if (k < 2 * nmem) sweep_body<1, MIX, 0, true, false, 0, true>(p, b, nblk, false, lds);
    else sweep_body<2, MIX, 0, true, false, 0, true>(p, b, nblk, false, lds);
}

template <bool CMP>
__global__ __launch_bounds__(256) void ens_update_kernel(const UpdateArgs* __restrict__ members,
                                                        const int* __restrict__ first, int nmem)
{
    const int m = entry_of(first, nmem, blockIdx.x);
    const UpdateArgs a = members[m];
    const long c = (long)(blockIdx.x - first[m]) * 256 + threadIdx.x;
    double t[5];
    if (c < a.plane) update_cell<CMP>(a, c, t);
}

hipError_t launch_ens_small_step(const SweepArgs* faces, const int* ffirst, int nfblk, const UpdateArgs* upd,
                                 const int* ufirst, int nublk, int nmem, bool mixed, bool compensated, hipStream_t s)
{
    if (nmem <= 0 || nfblk <= 0 || nublk <= 0 || (compensated && !mixed)) return hipErrorInvalidValue;
    const dim3 fg((unsigned)nfblk), ug((unsigned)nublk), block(256);
    if (mixed) hipLaunchKernelGGL(ens_faces_kernel<true>, fg, block, 0, s, faces, ffirst, nmem);
    else hipLaunchKernelGGL(ens_faces_kernel<false>, fg, block, 0, s, faces, ffirst, nmem);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (compensated) hipLaunchKernelGGL(ens_update_kernel<true>, ug, block, 0, s, upd, ufirst, nmem);
    else hipLaunchKernelGGL(ens_update_kernel<false>, ug, block, 0, s, upd, ufirst, nmem);
    return hipGetLastError();
}

static const int* tile_shape(int dir, int tile, bool mixed) { return mixed ? kTiles[dir][tile] : kTilesPair[dir][tile]; }

bool small_step_ok(int nc, bool mixed)
{
    bool ok = nc >= 16 && !(mixed && nc % 2) && nc <= (mixed ? kSmallNcMixed : kSmallNc);
    for (int d = 0; d < 3; d++) {
        const int* t = tile_shape(d, 0, mixed);
        ok = ok && t[0] + 3 <= nc && t[1] <= nc && t[2] <= nc;
    }
    return ok;
}

// segments of at most `most` chunks of CN faces: in equal parts where CN divides
// the line (the segment then divides the grid too: sweep_exact)
static int equal_parts(int nc, int CN, int most)
{
    const int lchunks = cdiv(nc, CN);
    int parts = cdiv(lchunks, most);
    if (nc % CN == 0)
        while (lchunks % parts) parts++;
    return cdiv(lchunks, parts) * CN;
}

// Faces per workgroup of faces_kernel along the sweep axis.  A workgroup's chunks
// pay one start (FP64: the ring's window, half a chunk; mixed: a quarter) and the
// launch ends a quarter of a workgroup's time after the slots run dry, so longer segments
// pay on larger grids only (us per step at 1 / 2 / 4 / 8 chunks, FP64: 32^3 29 /
// 32 / 35 / 51, 64^3 135 / 125 / 122 / 123, 128^3 898 / 805 / 773 / 765; mixed:
// 32^3 31 / 34 / 49 / 82, 128^3 813 / 793 / 762 / 767).  A member of an
// ensemble answers for its share of the launch's end.
static int faces_seg_len(int dir, int nc, int slots, double share, bool mixed)
{
    const int* t = tile_shape(dir, 0, mixed);
    const long pencils = (long)cdiv(nc, t[1]) * cdiv(nc, t[2]);
    const double start = mixed ? 0.25 : 0.5;
    int best = t[0];
    double cost = -1.0;
    for (int k = 1; k <= 8; k++) {
        const int seg = equal_parts(nc, t[0], k);
        if (seg > nc) break;
        const double chunks = seg / t[0] + start;
        const double c = (double)(pencils * sweep_nseg(nc, seg)) / slots * chunks + 0.25 * share * chunks;
        if (cost < 0.0 || c < cost) {
            cost = c;
            best = seg;
        }
    }
    return best;
}

SweepArgs faces_args(const SweepArgs& a, double* F, int dir, int slots, double share, bool mixed)
{
    SweepArgs f = a;
    f.tile = 0;
    f.mode = 0;
    f.dW = F + (long)dir * 5 * a.plane;
    f.seg = faces_seg_len(dir, a.nc, slots, share, mixed);
    f.nseg = sweep_nseg(a.nc, f.seg);
    return f;
}

int faces_blocks(int dir, const SweepArgs& f, bool mixed)
{
    const int* t = tile_shape(dir, 0, mixed);
    return cdiv(f.nc, t[1]) * cdiv(f.nc, t[2]) * f.nseg;
}

UpdateArgs update_args(const SweepArgs& a, const double* F)
{
    return {a.W, a.Wout, F, a.cmp_in, a.cmp_out, a.plane, a.nc, a.inv_dx, 0.0, 0.0, a.dx, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
}

hipError_t launch_small_step(const SweepArgs& a, double* F, const StepCfl* cfl, int slots, bool mixed, hipStream_t s)
{
    if (!small_step_ok(a.nc, mixed) || !F || (a.cmp_out != nullptr) != (a.cmp_in != nullptr) || (a.cmp_out && !mixed))
        return hipErrorInvalidValue;
    FaceArgs f{};
    for (int d = 0; d < 3; d++) {
        f.dir[d] = faces_args(a, F, d, slots, 1.0, mixed);
        f.first[d + 1] = f.first[d] + faces_blocks(d, f.dir[d], mixed);
    }
    const dim3 grid(f.first[3]), block(256);
    if (mixed) hipLaunchKernelGGL(faces_kernel<true>, grid, block, 0, s, f);
    else hipLaunchKernelGGL(faces_kernel<false>, grid, block, 0, s, f);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    UpdateArgs u = update_args(a, F);
    if (cfl) {
        u.gam = cfl->gam;
        u.cfl = cfl->cfl;
        u.partial = cfl->partial;
        u.dt = cfl->dt;
        u.vmax = cfl->vmax;
        u.hist = cfl->hist;
        u.bad = cfl->bad;
        u.ticket = cfl->ticket;
    }
    // with the CFL one maximum and one ticket per block: two blocks per CU
    const long all = (a.plane + 255) / 256, blocks = cfl && all > 512 ? 512 : all;
    static_assert(512 <= kCflBlocks, "a partial maximum per block");
    if (a.cmp_out) hipLaunchKernelGGL(step_update_kernel<true>, dim3((unsigned)blocks), block, 0, s, u);
    else hipLaunchKernelGGL(step_update_kernel<false>, dim3((unsigned)blocks), block, 0, s, u);
    return hipGetLastError();
}

bool sweep_tile_ok(int dir, int tile, int nc)
{
    // Any grid size: the pencils and segments of the last tiles reach past nc
    // (those lines and faces are computed with wrapped cells and not written).
    // Every wrapped index must stay in [-nc, 2nc), the range wrapi handles:
    // stencils reach CN + 2 cells before a segment and past the grid's end,
    // pencils one line past a tile.
    if (dir < 0 || dir > 2 || tile < 0 || tile >= kTileVariants) return false;
    const int CN = kTiles[dir][tile][0], CA = kTiles[dir][tile][1], CB = kTiles[dir][tile][2];
    return CN + 3 <= nc && CA <= nc && CB <= nc;
}

int sweep_first_tile(int dir, int nc)
{
    for (int v = 0; v < kTileVariants; v++)
        if (sweep_tile_ok(dir, v, nc)) return v;
    return -1;
}

bool sweep_grid_ok(int nc)
{
    return nc >= 16 && sweep_first_tile(0, nc) >= 0 && sweep_first_tile(1, nc) >= 0 && sweep_first_tile(2, nc) >= 0;
}

int sweep_seg_len(int dir, int nc, int tile, int slots, bool mixed)
{
    // faces per workgroup along the sweep axis (a multiple of CN); a segment
    // costs seg/CN chunks plus one lead-in chunk (the face before the segment).
    if (!sweep_tile_ok(dir, tile, nc)) return 0;
    const int* t = tile_shape(dir, tile, mixed);
    const int CN = t[0], CA = t[1], CB = t[2];
    const long pencils = (long)cdiv(nc, CA) * cdiv(nc, CB);
    const int lchunks = cdiv(nc, CN);  // chunks of a whole line
    if (slots > 0) {
        // one grid: the length with the fewest chunk-times, counting rounds of
        // `slots` concurrent workgroups; the longer segment on ties
        int best = lchunks * CN;
        long best_cost = -1;
        for (int parts = 1;; parts *= 2) {
            const int seg = cdiv(lchunks, parts) * CN;
            if (seg == nc - 1) continue;  // its last workgroups run past one wrap (sweep_seg_most)
            const long blocks = pencils * cdiv(nc, seg);
            const long cost = (blocks + slots - 1) / slots * (seg / CN + 1);
            if (best_cost < 0 || cost < best_cost) {
                best_cost = cost;
                best = seg;
            }
            if (seg == CN) break;
        }
        return best;
    }
    return lchunks * CN;  // an ensemble's members: whole lines, or sweep_seg_most
}

int sweep_seg_most(int dir, int nc, int tile, int most, bool mixed)
{
    if (!sweep_tile_ok(dir, tile, nc) || most < 1) return 0;
    const int CN = tile_shape(dir, tile, mixed)[0];
    const int seg = equal_parts(nc, CN, most);
    // a last segment of one face whose workgroups run on to cell 2 nc, one past
    // what a single wrap reaches (33^3 in segments of 32, 17^3 in segments of 16):
    // the next shorter ones
    return seg == nc - 1 ? equal_parts(nc, CN, seg / CN - 1) : seg;
}

template <int DIR, int V>
static hipError_t launch_tile(const SweepArgs& a, bool mixed, hipStream_t s)
{
    const int* t = tile_shape(DIR, V, mixed);
    const int CN = t[0], CA = t[1], CB = t[2];
    if (!sweep_tile_ok(DIR, V, a.nc) || a.seg <= 0 || a.seg % CN || a.nseg != cdiv(a.nc, a.seg))
        return hipErrorInvalidValue;
    const long nblk = (long)cdiv(a.nc, CA) * cdiv(a.nc, CB) * a.nseg;
    // the compensated update is the mixed z sweep's (an FP64 context has no carry)
    if ((a.cmp_out != nullptr) != (a.cmp_in != nullptr) || (a.cmp_out && !mixed)) return hipErrorInvalidValue;
    const bool gen = !sweep_exact(DIR, V, a.nc, a.seg, mixed);  // some workgroup reaches past the grid
    const bool cmp = a.cmp_out && a.mode == 2;
    const dim3 grid((unsigned)nblk), block(256);
    if (mixed) {
        if constexpr (DIR == 2) {
            if (cmp) {
                if (gen) hipLaunchKernelGGL((sweep_kernel<DIR, true, V, true, 1>), grid, block, 0, s, a);
                else hipLaunchKernelGGL((sweep_kernel<DIR, true, V, false, 1>), grid, block, 0, s, a);
                return hipGetLastError();
            }
        }
        if (gen) hipLaunchKernelGGL((sweep_kernel<DIR, true, V, true, 0>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((sweep_kernel<DIR, true, V, false, 0>), grid, block, 0, s, a);
    } else {
        if (gen) hipLaunchKernelGGL((sweep_kernel<DIR, false, V, true, 0>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((sweep_kernel<DIR, false, V, false, 0>), grid, block, 0, s, a);
    }
    return hipGetLastError();
}

template <int DIR>
static hipError_t launch_dir(const SweepArgs& a, bool mixed, hipStream_t s)
{
    static_assert(kTileVariants == 3, "one case per tile variant");
    switch (a.tile) {
    case 0: return launch_tile<DIR, 0>(a, mixed, s);
    case 1: return launch_tile<DIR, 1>(a, mixed, s);
    case 2: return launch_tile<DIR, 2>(a, mixed, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_sweep(int dir, const SweepArgs& a, bool mixed, hipStream_t s)
{
    if (dir == 0) return launch_dir<0>(a, mixed, s);
    if (dir == 1) return launch_dir<1>(a, mixed, s);
    if (dir == 2) return launch_dir<2>(a, mixed, s);
    return hipErrorInvalidValue;
}

int sweep_blocks(int dir, int nc, int tile, int seg, bool mixed)
{
    if (!sweep_tile_ok(dir, tile, nc) || seg <= 0) return 0;
    const int* t = tile_shape(dir, tile, mixed);
    return cdiv(nc, t[1]) * cdiv(nc, t[2]) * cdiv(nc, seg);
}

int sweep_chunks(int dir, int tile, int seg, bool mixed) { return seg / tile_shape(dir, tile, mixed)[0]; }

bool sweep_exact(int dir, int tile, int nc, int seg, bool mixed)
{
    if (!sweep_tile_ok(dir, tile, nc) || seg <= 0) return false;
    const int* t = tile_shape(dir, tile, mixed);
    return nc % t[1] == 0 && nc % t[2] == 0 && nc % seg == 0;
}

template <int DIR, int V>
static hipError_t launch_ens_tile(const SweepArgs* members, const int* first, int nmem, int nblk, bool mixed,
                                  bool exact, bool cmp, hipStream_t s)
{
    const dim3 grid((unsigned)nblk), block(256);
    if (mixed) {
        if constexpr (DIR == 2) {
            if (cmp) {
                if (exact) hipLaunchKernelGGL((ens_sweep_kernel<DIR, true, V, false, 1>), grid, block, 0, s, members, first, nmem);
                else hipLaunchKernelGGL((ens_sweep_kernel<DIR, true, V, true, 1>), grid, block, 0, s, members, first, nmem);
                return hipGetLastError();
            }
        }
        if (exact) hipLaunchKernelGGL((ens_sweep_kernel<DIR, true, V, false, 0>), grid, block, 0, s, members, first, nmem);
        else hipLaunchKernelGGL((ens_sweep_kernel<DIR, true, V, true, 0>), grid, block, 0, s, members, first, nmem);
    } else {
        if (exact) hipLaunchKernelGGL((ens_sweep_kernel<DIR, false, V, false, 0>), grid, block, 0, s, members, first, nmem);
        else hipLaunchKernelGGL((ens_sweep_kernel<DIR, false, V, true, 0>), grid, block, 0, s, members, first, nmem);
    }
    return hipGetLastError();
}

template <int DIR>
static hipError_t launch_ens_dir(int tile, const SweepArgs* members, const int* first, int nmem, int nblk, bool mixed,
                                 bool exact, bool cmp, hipStream_t s)
{
    switch (tile) {
    case 0: return launch_ens_tile<DIR, 0>(members, first, nmem, nblk, mixed, exact, cmp, s);
    case 1: return launch_ens_tile<DIR, 1>(members, first, nmem, nblk, mixed, exact, cmp, s);
    case 2: return launch_ens_tile<DIR, 2>(members, first, nmem, nblk, mixed, exact, cmp, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_ens_sweep(int dir, int tile, const SweepArgs* members, const int* first, int nmem, int nblk,
                            bool mixed, bool exact, bool compensated, hipStream_t s)
{
    if (nmem <= 0 || nblk <= 0 || (compensated && !mixed)) return hipErrorInvalidValue;
    if (dir == 0) return launch_ens_dir<0>(tile, members, first, nmem, nblk, mixed, exact, compensated, s);
    if (dir == 1) return launch_ens_dir<1>(tile, members, first, nmem, nblk, mixed, exact, compensated, s);
    if (dir == 2) return launch_ens_dir<2>(tile, members, first, nmem, nblk, mixed, exact, compensated, s);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// CFL: dt = cfl dx / max(|U| + sqrt(gam p / rho)) over all cells
// (timestep, update.cpp:1031-1054).  A block maximum goes to partial[]; a
// non-physical cell (rho <= 0, p <= 0 or not finite) records -1 instead.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void cfl_partial_kernel(const double* __restrict__ W, long plane, double gam,
                                                          double* partial)
{
    cfl_cells(W, plane, gam, (long)blockIdx.x * blockDim.x, (long)gridDim.x * blockDim.x, partial + blockIdx.x);
}

__global__ __launch_bounds__(256) void cfl_final_kernel(const double* partial, int n, double cfl, double dx,
                                                        double* dt, double* vmax, int* bad, double* hist)
{
    cfl_reduce(partial, n, cfl, dx, dt, vmax, bad, hist);
}

__global__ void set_scalar_kernel(double* p, double v)
{
    if (threadIdx.x == 0) *p = v;
}
hipError_t launch_set_scalar(double* p, double v, hipStream_t s)
{
    hipLaunchKernelGGL(set_scalar_kernel, dim3(1), dim3(64), 0, s, p, v);
    return hipGetLastError();
}

hipError_t launch_cfl(const double* W, long plane, double gam, double cfl, double dx, double* partial, double* dt,
                      double* vmax, int* bad, double* hist, hipStream_t s)
{
    hipLaunchKernelGGL(cfl_partial_kernel, dim3(kCflBlocks), dim3(256), 0, s, W, plane, gam, partial);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(cfl_final_kernel, dim3(1), dim3(256), 0, s, partial, kCflBlocks, cfl, dx, dt, vmax, bad, hist);
    return hipGetLastError();
}

// Ensemble CFL: kEnsCflBlocks blocks per member reduce max(|U|+c) of that
// member's cells into partial[m * kEnsCflBlocks + b]; one block per member then
// writes dt = cfl dx / max (0 and the flag when a state is non-physical).
__global__ __launch_bounds__(256) void ens_cfl_partial_kernel(const CflArgs* __restrict__ members, double* partial)
{
    const int m = blockIdx.x / kEnsCflBlocks, b = blockIdx.x % kEnsCflBlocks;
    const CflArgs a = members[m];
    cfl_cells(a.W, a.plane, a.gam, (long)b * blockDim.x, (long)kEnsCflBlocks * blockDim.x, partial + blockIdx.x);
}

__global__ __launch_bounds__(256) void ens_cfl_final_kernel(const CflArgs* __restrict__ members, const double* partial)
{
    const CflArgs a = members[blockIdx.x];
    cfl_reduce(partial + (long)blockIdx.x * kEnsCflBlocks, kEnsCflBlocks, a.cfl, a.dx, a.dt, a.vmax, a.bad);
}

hipError_t launch_ens_cfl(const CflArgs* members, int nmem, double* partial, hipStream_t s)
{
    if (nmem <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(ens_cfl_partial_kernel, dim3((unsigned)(nmem * kEnsCflBlocks)), dim3(256), 0, s, members,
                       partial);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(ens_cfl_final_kernel, dim3((unsigned)nmem), dim3(256), 0, s, members, partial);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Layout conversion.  pack fills the host layout's 3 ghost layers per face
// periodically: ghost(i) = cell(((i-3) mod nc) + 3) on every axis (the
// single-domain result of HaloTransfer, update.cpp:855-1029).
// ---------------------------------------------------------------------------
__global__ void unpack_kernel(const double* __restrict__ padded, double* __restrict__ W, int nc)
{
    const long plane = (long)nc * nc * nc;
    const int nt = nc + 6;
    const long ntp = (long)nt * nt * nt;
    for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < 5 * plane; c += (long)gridDim.x * blockDim.x) {
        const int q = (int)(c / plane);
        const long r = c - q * plane;
        const int k = (int)(r % nc), i = (int)((r / nc) % nc), j = (int)(r / ((long)nc * nc));
        W[c] = padded[q * ntp + ((long)(j + 3) * nt + (i + 3)) * nt + (k + 3)];
    }
}

__global__ void pack_kernel(const double* __restrict__ W, double* __restrict__ padded, int nc)
{
    const long plane = (long)nc * nc * nc;
    const int nt = nc + 6;
    const long ntp = (long)nt * nt * nt;
    for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < 5 * ntp; c += (long)gridDim.x * blockDim.x) {
        const int q = (int)(c / ntp);
        const long r = c - q * ntp;
        const int k = (int)(r % nt), i = (int)((r / nt) % nt), j = (int)(r / ((long)nt * nt));
        const int jj = (j - 3 + nc) % nc, ii = (i - 3 + nc) % nc, kk = (k - 3 + nc) % nc;
        padded[c] = W[q * plane + ((long)jj * nc + ii) * nc + kk];
    }
}

static unsigned grid_for(long n, int block)
{
    long g = (n + block - 1) / block;
    if (g > 65536) g = 65536;
    if (g < 1) g = 1;
    return (unsigned)g;
}

hipError_t launch_unpack(const double* padded, double* W, int nc, hipStream_t s)
{
    const long n = 5L * nc * nc * nc;
    hipLaunchKernelGGL(unpack_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, padded, W, nc);
    return hipGetLastError();
}

hipError_t launch_pack(const double* W, double* padded, int nc, hipStream_t s)
{
    const long nt = nc + 6;
    const long n = 5L * nt * nt * nt;
    hipLaunchKernelGGL(pack_kernel, dim3(grid_for(n, 256)), dim3(256), 0, s, W, padded, nc);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Pointwise kernels for parity checks of the device math
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(64) void flux_batch_kernel(long n, const double* __restrict__ in, const double* __restrict__ tau, double dt,
                                  double dx, Gas<T> g, double* __restrict__ F)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double* v = in + 50 * i;
    T WL[5], WR[5], Wl[5], Wr[5], D[6][5], Fo[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
        WL[q] = (T)v[q];
        WR[q] = (T)v[5 + q];
        Wl[q] = (T)v[10 + q];
        Wr[q] = (T)v[15 + q];
#pragma unroll
        for (int d = 0; d < 6; d++) D[d][q] = (T)v[20 + 5 * d + q];
    }
    gks_flux_tf<T, T>(WL, WR, Wl, Wr, D, (T)tau[i], (T)dt, (T)dx, g, Fo);
#pragma unroll
    for (int q = 0; q < 5; q++) F[5 * i + q] = (double)Fo[q];
}

// FP64: two threads per face, the sweeps' flux (gkm_pair.hpp)
struct BatchSide {
    double s[5], c[5], n[5], t[2][5];
    __device__ double S(int q) const { return s[q]; }
    __device__ double C(int q) const { return c[q]; }
    __device__ double N(int q) const { return n[q]; }
    __device__ double T(int k, int q) const { return t[k][q]; }
};
__global__ __launch_bounds__(64) void flux_batch_pair_kernel(long n, const double* __restrict__ in,
                                                             const double* __restrict__ tau, double dt, double dx,
                                                             GasK g, double* __restrict__ F)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int side = (int)(t & 1);
    const bool live = (t >> 1) < n;
    const long i = live ? t >> 1 : n - 1;  // lanes past the end repeat the last face: the pair exchange needs them
    const double* v = in + 50 * i;
    BatchSide b;
#pragma unroll
    for (int q = 0; q < 5; q++) {
        // side 1 in its mirrored frame: slots 2 and 3 and the tangential
        // directions change places, slot 1 and the normal direction their sign
        const int p = side && (q == 2 || q == 3) ? 5 - q : q;
        const double m = side && q == 1 ? -1.0 : 1.0;
        b.c[q] = m * v[5 * side + p];
        b.s[q] = m * v[10 + 5 * side + p];
        b.n[q] = (side ? -m : m) * v[20 + 5 * side + p];
        b.t[0][q] = m * v[(side ? 45 : 30) + p];
        b.t[1][q] = m * v[(side ? 35 : 40) + p];
    }
    double Fo[5];
    gks_flux_pair(b, tau[i], dt, dx, g, PairSwap{}, Fo);
    if (live && side == 0)
#pragma unroll
        for (int q = 0; q < 5; q++) F[5 * i + q] = Fo[q];
}

__global__ __launch_bounds__(64) void flux_batch_mixed_kernel(long n, const double* __restrict__ in,
                                                              const double* __restrict__ tau, double dt, double dx,
                                                              Gas<double> g, double* __restrict__ F)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double* v = in + 50 * i;
    double WL[5], WR[5], Wl[5], Wr[5], D[6][5], Fo[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
        WL[q] = v[q];
        WR[q] = v[5 + q];
        Wl[q] = v[10 + q];
        Wr[q] = v[15 + q];
#pragma unroll
        for (int d = 0; d < 6; d++) D[d][q] = v[20 + 5 * d + q];
    }
    gks_flux_tf<double, float>(WL, WR, Wl, Wr, D, tau[i], dt, dx, g, Fo);
#pragma unroll
    for (int q = 0; q < 5; q++) F[5 * i + q] = Fo[q];
}

template <typename T>
__global__ __launch_bounds__(64) void weno_batch_kernel(long n, const double* __restrict__ in, Gas<T> g, double* __restrict__ out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    T S[6][5], Wl[5], Wr[5];
#pragma unroll
    for (int s = 0; s < 6; s++)
#pragma unroll
        for (int q = 0; q < 5; q++) S[s][q] = (T)in[30 * i + 5 * s + q];
    weno5<T>(S, g, Wl, Wr);
#pragma unroll
    for (int q = 0; q < 5; q++) {
        out[10 * i + q] = (double)Wl[q];
        out[10 * i + 5 + q] = (double)Wr[q];
    }
}

__global__ __launch_bounds__(64) void weno_batch_mixed_kernel(long n, const double* __restrict__ in, Gas<double> g,
                                                              double* __restrict__ out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double S[6][5], Wl[5], Wr[5];
#pragma unroll
    for (int s = 0; s < 6; s++)
#pragma unroll
        for (int q = 0; q < 5; q++) S[s][q] = in[30 * i + 5 * s + q];
    weno5_mixed(S, g, Wl, Wr);
#pragma unroll
    for (int q = 0; q < 5; q++) {
        out[10 * i + q] = Wl[q];
        out[10 * i + 5 + q] = Wr[q];
    }
}


hipError_t launch_flux_batch(long n, const double* in, const double* tau, double dt, double dx, const Gas<double>& g,
                             int precision, double* F, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const unsigned blocks = (unsigned)((n + 63) / 64);
    if (precision == 0)
        hipLaunchKernelGGL(flux_batch_pair_kernel, dim3((unsigned)((2 * n + 63) / 64)), dim3(64), 0, s, n, in, tau, dt,
                           dx, gas_const(g), F);
    else if (precision == 1)
        hipLaunchKernelGGL(flux_batch_mixed_kernel, dim3(blocks), dim3(64), 0, s, n, in, tau, dt, dx, g, F);
    else
        hipLaunchKernelGGL(flux_batch_kernel<float>, dim3(blocks), dim3(64), 0, s, n, in, tau, dt, dx, to_f32(g), F);
    return hipGetLastError();
}

hipError_t launch_weno_batch(long n, const double* in, const Gas<double>& g, int precision, double* out, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    const unsigned blocks = (unsigned)((n + 63) / 64);
    if (precision == 0)
        hipLaunchKernelGGL(weno_batch_kernel<double>, dim3(blocks), dim3(64), 0, s, n, in, g, out);
    else if (precision == 1)
        hipLaunchKernelGGL(weno_batch_mixed_kernel, dim3(blocks), dim3(64), 0, s, n, in, g, out);
    else
        hipLaunchKernelGGL(weno_batch_kernel<float>, dim3(blocks), dim3(64), 0, s, n, in, to_f32(g), out);
    return hipGetLastError();
}

}  // namespace gkm
