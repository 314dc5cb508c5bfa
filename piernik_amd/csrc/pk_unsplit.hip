// pk_unsplit.hip -- gfx950 kernels of the unsplit Riemann stage
// (solve_cg_ub / solve_cg_u of src/scheme/unsplit_schemes/, one RK stage).
//
// k_unsplit_flux_tile: the interface fluxes of the transverse-interior
// pencils along one direction, from tiles of TP pencils x TS cells.  A lane
// computes the primitives (sweep order) and limited slopes of its cell once,
// the face states go through LDS, and the lane of cell c evaluates HLLD + GLM
// or HLLC at c+1/2, exactly as interpol and riemann_wrap do for that
// interface (unsplit_mag_modules.F90:166-209, solve_cg_unsplit.F90:157-187).
// Lanes run x fastest, so y and z loads are coalesced.
//
// k_unsplit_update: one lane per interior cell.  The flux differences of
// x, then y, then z are added to the base state (apply_flux and update_psi,
// unsplit_mag_modules.F90:211-328), then apply_source's passes run over the
// directions in turn (unsplit_source.F90:42-132): +0 from the vanishing
// internal sources and, at the last stage, care_for_positives in that
// direction's sweep order.  Ghost cells are not written: update_boundaries
// replaces them after every stage.
//
// k_unsplit_fused_tile: both in one pass per direction, for stages whose
// output is not their input (the two RK2 stages): the flux tile adds each
// cell's flux difference to a running sum kept in the output buffer, and the
// last direction's pass runs the sources.  Same operands in the same order,
// so the same bits, without writing and re-reading the flux arrays.
//
// Built without FMA contraction (namespace pk): bit-identical to the
// oracle's unsplit driver.  pk_unsplit_fast.hip builds the same source with
// contraction and fast division into namespace pk_fast.
#include <hip/hip_runtime.h>
#include "pk_math.hpp"
#include "pk_mass.hpp"
#include "pk_kernels.hpp"
#include "pk_unsplit.hpp"

namespace PK_KNS {

using pk::UnsplitArgs;

#include "pk_tile.hpp"

namespace {

// plane_of for a direction that is a loop's variable
__device__ __forceinline__ int uplane(int dir, int k)
{
    return dir == 0 ? plane_of<0>(k) : (dir == 1 ? plane_of<1>(k) : plane_of<2>(k));
}

// Tile of TP pencils x TS cells along DIR, lanes x fastest.  The lane of
// cell c evaluates the Riemann flux at c+1/2 from its right face state and
// the left face state of cell c+1: l = q(c) + 0.5*limit(q(c)-q(c-1),
// q(c+1)-q(c)) and r = q(c+1) - 0.5*limit(...), the operands and operations
// of the reference's per-interface formula.  The tile starts one cell before
// the left cell of its first interface; TS-3 fluxes per tile, row c+1 of F
// holding the flux at c+1/2.
template <int DIR, class P, int LIM>
__global__ __launch_bounds__(256) void k_unsplit_flux_tile(const UnsplitArgs a, double *__restrict__ F, int TP,
                                                           int TS, int chunks)
{
    constexpr int NV = P::NV;
    constexpr int d1 = (DIR == 0) ? 1 : 0;
    constexpr int d2 = (DIR == 2) ? 1 : 2;
    extern __shared__ double lds[];
    double *A = lds;                   // primitives
    double *B = lds + NV * blockDim.x; // left face states
    const int nt = blockDim.x;
    const int t = threadIdx.x;
    const int bid = (int)pk::xcd_order();
    int p, sl, tm, tp;
    if (DIR == 0) {
        p = small_div(t, TS);
        sl = t - p * TS;
        tm = t - 1;
        tp = t + 1;
    } else {
        sl = small_div(t, TP);
        p = t - sl * TP;
        tm = t - TP;
        tp = t + TP;
    }
    tm = tm < 0 ? 0 : tm;
    tp = tp >= nt ? nt - 1 : tp;
    const int chunk = bid % chunks;
    const int ptile = bid / chunks;
    const int n1 = a.n[d1];
    const int npen = n1 * a.n[d2];
    const int pf = ptile * TP + p;
    const bool pvalid = t < TP * TS && pf < npen;
    const int pfc = pf < npen ? pf : npen - 1;
    const int out = TS - 3;
    const int c0 = a.g[DIR] - 1 + chunk * out;  // left cell of the tile's first interface
    const int cs = c0 - 1 + sl;                 // this lane's cell (the tile starts at c0 - 1)
    const int ng = a.ng[DIR];
    const int csc = cs < 0 ? 0 : (cs >= ng ? ng - 1 : cs);
    int xyz[3];
    xyz[DIR] = csc;
    const int e0 = (ptile * TP) / n1;  // the tile's first pencil: uniform, the lanes step on from it
    int e1 = ptile * TP - e0 * n1 + (pfc - ptile * TP), e2 = e0;
    if (n1 >= TP) {
        if (e1 >= n1) e1 -= n1, e2++;
    } else {
        e2 += e1 / n1;
        e1 = e1 % n1;
    }
    xyz[d1] = a.g[d1] + e1;
    xyz[d2] = a.g[d2] + e2;
    const long long idx = (long long)xyz[0] + (long long)a.sy * xyz[1] + (long long)a.sz * xyz[2];

    double W[NV], q[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) W[k] = a.src[(long long)plane_of<DIR>(k) * a.sv + idx];
    prim<P>(W, a.gam_1, q);
    lds_put<NV>(A, t, q);
    __syncthreads();
    double fp[NV];
    {
        double qm[NV], qp[NV], fm[NV];
        lds_get<NV>(A, tm, qm);
        lds_get<NV>(A, tp, qp);
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const int lim = (LIM >= 0) ? LIM : ((v < 5) ? a.lim : a.limb);
            const double h = 0.5 * limit(lim, q[v] - qm[v], qp[v] - q[v]);
            fp[v] = q[v] + h;  // right face of this cell
            fm[v] = q[v] - h;  // left face of this cell
        }
        lds_put<NV>(B, t, fm);
    }
    __syncthreads();
    // the flux at cs+1/2, row cs+1, for interfaces g-1/2 .. g+n-1/2
    const bool own = pvalid && sl >= 1 && sl < 1 + out && cs >= a.g[DIR] - 1 && cs <= a.g[DIR] + a.n[DIR] - 1;
    if (!own) return;
    double fr[NV], f[NV];
    lds_get<NV>(B, tp, fr);
    if constexpr (P::MAG)
        flux_hlld(fp, fr, a.gam, a.ch, f);
    else
        flux_hllc(fp, fr, a.gam, f);
    const long long st = (DIR == 0) ? 1ll : ((DIR == 1) ? (long long)a.sy : (long long)a.sz);
    const long long row = idx + st;
#pragma unroll
    for (int k = 0; k < NV; k++) F[(long long)plane_of<DIR>(k) * a.sv + row] = f[k];
}

// Flux along DIR and its difference in one tile (dst != src).  The tile
// starts two cells before its first updated cell (TS-4 per tile); lanes 1 ..
// TS-3 evaluate the flux at their cell's right face as k_unsplit_flux_tile
// does, and the lane of cell c adds coef*(F(c-1/2) - F(c+1/2)), the left
// flux from its neighbour through LDS, to the cell's running sum.  The sum
// starts from base at the first active direction and waits in dst between
// directions, each cell read and written by its own lane only; after the
// last active direction the source passes run and dst holds the stage's
// result (interior cells; its ghosts are left as they are, and read through
// their pre-images: a.wrap).  The operands and their order are those of
// k_unsplit_update, so the result is the same bit for bit, without the flux
// arrays.
// Bound by memory where it adds to dst (read src and dst, write dst: 90 us at
// the copy rate for 128^3 MHD), by FP64 issue and memory both along x.  Lane-
// major LDS (pk_tile.hpp), chunks of equal length and no images: the passes of
// a 128^3 MHD block along x, y, z took 134, 141, 157 us with 4 x 64 and 8 x 32
// tiles, images and [variable][lane] LDS; 101, 116, 129 us now.
template <int DIR, class P, int LIM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_unsplit_fused_tile(const UnsplitArgs a, int TP, int TS, int chunks,
                                                            int first, int last)
{
    constexpr int NV = P::NV;
    constexpr int d1 = (DIR == 0) ? 1 : 0;
    constexpr int d2 = (DIR == 2) ? 1 : 2;
    extern __shared__ double lds[];
    double *A = lds;                    // primitives, then fluxes
    double *B = lds + NV * blockDim.x;  // left face states
    const int nt = blockDim.x;
    const int t = threadIdx.x;
    const int bid = (int)pk::xcd_order();
    int p, sl, tm, tp;
    if (DIR == 0) {
        p = small_div(t, TS);
        sl = t - p * TS;
        tm = t - 1;
        tp = t + 1;
    } else {
        sl = small_div(t, TP);
        p = t - sl * TP;
        tm = t - TP;
        tp = t + TP;
    }
    tm = tm < 0 ? 0 : tm;
    tp = tp >= nt ? nt - 1 : tp;
    const int chunk = bid % chunks;
    const int ptile = bid / chunks;
    const int n1 = a.n[d1];
    const int npen = n1 * a.n[d2];
    const int pf = ptile * TP + p;
    const bool pvalid = t < TP * TS && pf < npen;
    const int pfc = pf < npen ? pf : npen - 1;
    const int out = TS - 4;
    const int c0 = a.g[DIR] + chunk * out;  // the tile's first updated cell
    const int cs = c0 - 2 + sl;             // this lane's cell
    const int ng = a.ng[DIR];
    int csc = cs < 0 ? 0 : (cs >= ng ? ng - 1 : cs);
    if (a.wrap) csc = wrap_cell(csc, a.g[DIR], a.n[DIR]);
    int xyz[3];
    xyz[DIR] = csc;
    const int e0 = (ptile * TP) / n1;  // the tile's first pencil: uniform, the lanes step on from it
    int e1 = ptile * TP - e0 * n1 + (pfc - ptile * TP), e2 = e0;
    if (n1 >= TP) {
        if (e1 >= n1) e1 -= n1, e2++;
    } else {
        e2 += e1 / n1;
        e1 = e1 % n1;
    }
    xyz[d1] = a.g[d1] + e1;
    xyz[d2] = a.g[d2] + e2;
    const long long idx = (long long)xyz[0] + (long long)a.sy * xyz[1] + (long long)a.sz * xyz[2];

    double W[NV], q[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) W[k] = a.src[(long long)plane_of<DIR>(k) * a.sv + idx];
    if constexpr (P::MAG) W[8] = W[8] * a.src_fac;
    prim<P>(W, a.gam_1, q);
    lds_put<NV>(A, t, q);
    __syncthreads();
    double fp[NV];
    {
        double qm[NV], qp[NV], fm[NV];
        lds_get<NV>(A, tm, qm);
        lds_get<NV>(A, tp, qp);
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const int lim = (LIM >= 0) ? LIM : ((v < 5) ? a.lim : a.limb);
            const double h = 0.5 * limit(lim, q[v] - qm[v], qp[v] - q[v]);
            fp[v] = q[v] + h;
            fm[v] = q[v] - h;
        }
        lds_put<NV>(B, t, fm);
    }
    __syncthreads();
    double f[NV];
    if (sl >= 1 && sl < TS - 2) {
        double fr[NV];
        lds_get<NV>(B, tp, fr);
        if constexpr (P::MAG)
            flux_hlld(fp, fr, a.gam, a.ch, f);
        else
            flux_hllc(fp, fr, a.gam, f);
    } else {
#pragma unroll
        for (int v = 0; v < NV; v++) f[v] = 0.0;
    }
    const bool upd = pvalid && sl >= 2 && sl < 2 + out && cs < a.g[DIR] + a.n[DIR];
    const long long ci = idx;  // an interior cell when upd: csc == cs
    double T[NV];
    if (upd) {
        const double *S = first ? a.base : a.dst;
#pragma unroll
        for (int v = 0; v < NV; v++) T[v] = S[(long long)v * a.sv + ci];
    }
    // every read of A (the primitives) came before the last barrier
    lds_put<NV>(A, t, f);
    __syncthreads();
    unsigned flags = 0u;
    double dmass = 0.0;
    if (upd) {
        if constexpr (P::MAG) {
            if (first) T[8] = T[8] * a.base_fac;
        }
        const double coef = (a.dt / a.dl[DIR]) * a.rk;
        double fl[NV];
        lds_get<NV>(A, tm, fl);
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int v = plane_of<DIR>(k);
            T[v] = T[v] + coef * (fl[k] - f[k]);
        }
        if (last) {
            for (int d = 0; d < 3; d++) {
                if (!a.has_dir[d]) continue;
                double Ws[NV];
#pragma unroll
                for (int kk = 0; kk < NV; kk++) Ws[kk] = T[uplane(d, kk)];
#pragma unroll
                for (int v = 0; v < 5; v++) Ws[v] = Ws[v] + 0.0;
                if (a.last) {
                    unsigned fl = 0u;
                    double dm = 0.0;
                    floors<P>(Ws, a.smalld, a.smallei, a.use_smalld, a.use_smallei, a.ei_flag, fl, dm);
                    flags |= fl;
                    dmass += dm;  // one cell's floor events, in the direction order
                }
#pragma unroll
                for (int kk = 0; kk < NV; kk++) T[uplane(d, kk)] = Ws[kk];
            }
            if constexpr (P::MAG) T[8] = T[8] * a.psi_fac;  // glmdamping after the stages (1 at the first stage)
        }
#pragma unroll
        for (int v = 0; v < NV; v++) a.dst[(long long)v * a.sv + ci] = T[v];
    }
    // last, a.last and a.dtslots are the same for every lane: the whole wave takes part
    if (last && a.last) pk::mass_add(a.dmass, dmass);
#if !PK_RELAXED
    if (last && a.dtslots) {  // timestep_fluid of the cells of the finished state
        const double huge = 1.7976931348623157e308;
        double mn[3] = {huge, huge, huge}, cmax = 0.0;
        if (upd) dt_cell<0, P>(a, T, mn, cmax);
        dt_reduce(a, mn, cmax, blockIdx.x);
    }
#endif
    if (upd && flags) atomicOr(a.flags, flags);
}

template <class P>
__global__ __launch_bounds__(256) void k_unsplit_update(const UnsplitArgs a, const double *__restrict__ F0,
                                                        const double *__restrict__ F1,
                                                        const double *__restrict__ F2)
{
    constexpr int NV = P::NV;
    const long long nx = a.n[0], nxy = nx * a.n[1];
    const long long total = nxy * a.n[2];
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned flags = 0u;
    double dmass = 0.0;
    if (e < total) {
        const int i = (int)(e % nx), j = (int)((e / nx) % a.n[1]), k = (int)(e / nxy);
        const long long idx =
            (long long)(i + a.g[0]) + (long long)a.sy * (j + a.g[1]) + (long long)a.sz * (k + a.g[2]);
        double T[NV];
#pragma unroll
        for (int v = 0; v < NV; v++) T[v] = a.base[(long long)v * a.sv + idx];
        const double *Fd[3] = {F0, F1, F2};
        const long long st[3] = {1, a.sy, a.sz};
        for (int d = 0; d < 3; d++) {
            if (!a.has_dir[d]) continue;
            const double coef = (a.dt / a.dl[d]) * a.rk;
            const double *F = Fd[d];
#pragma unroll
            for (int v = 0; v < NV; v++)
                T[v] = T[v] + coef * (F[(long long)v * a.sv + idx] - F[(long long)v * a.sv + idx + st[d]]);
        }
        for (int d = 0; d < 3; d++) {
            if (!a.has_dir[d]) continue;
            double W[NV];
#pragma unroll
            for (int kk = 0; kk < NV; kk++) W[kk] = T[uplane(d, kk)];
#pragma unroll
            for (int v = 0; v < 5; v++) W[v] = W[v] + 0.0;
            if (a.last) {
                unsigned fl = 0u;
                double dm = 0.0;
                floors<P>(W, a.smalld, a.smallei, a.use_smalld, a.use_smallei, a.ei_flag, fl, dm);
                flags |= fl;
                dmass += dm;
            }
#pragma unroll
            for (int kk = 0; kk < NV; kk++) T[uplane(d, kk)] = W[kk];
        }
#pragma unroll
        for (int v = 0; v < NV; v++) a.dst[(long long)v * a.sv + idx] = T[v];
    }
    if (a.last) pk::mass_add(a.dmass, dmass);
    if (flags) atomicOr(a.flags, flags);
}

// Tile of the flux kernels for npen pencils of span rows, ts - lost finished per
// tile.  Along x the fewest workgroups (full_tile); along y and z 8 x-consecutive
// pencils, 64 bytes a row, in equal chunks of at most 32 cells: these passes
// wait for memory, and other widths leave part of every line to another
// workgroup (three steps of a 128^3 MHD block with 7 x 36 in y and z 2550 us,
// with 8 x 30 in y 2454 - 2330, in both 2230; hydro 1034, 1008).
template <int DIR>
void unsplit_tile(int span, long long npen, int lost, int &TP, int &TS)
{
    if (DIR == 0) {
        pk::full_tile(span, npen, lost, true, TP, TS);
        return;
    }
    TP = 8;
    const int k = (span + 32 - lost - 1) / (32 - lost);
    TS = (span + k - 1) / k + lost;
}

template <int DIR, class P, int LIM>
hipError_t fused_tile(const UnsplitArgs &a, int first, int last, hipStream_t st)
{
    const int d1 = (DIR == 0) ? 1 : 0, d2 = (DIR == 2) ? 1 : 2;
    const long long npen = (long long)a.n[d1] * a.n[d2];
    int TP, TS;
    unsplit_tile<DIR>(a.n[DIR], npen, 4, TP, TS);
    const int chunks = (a.n[DIR] + (TS - 4) - 1) / (TS - 4);
    const int nt = (TP * TS + 63) / 64 * 64;
    const long long tiles = (npen + TP - 1) / TP * chunks;
    if (tiles < 1 || tiles > 0x7fffffffll) return hipErrorInvalidValue;
    const size_t shm = sizeof(double) * 2 * P::NV * nt;
    hipLaunchKernelGGL((k_unsplit_fused_tile<DIR, P, LIM>), dim3((unsigned)tiles), dim3(nt), shm, st, a, TP,
                       TS, chunks, first, last);
    return hipGetLastError();
}

template <int DIR, class P>
hipError_t fused_lim(const UnsplitArgs &a, int first, int last, hipStream_t st)
{
    if (a.lim == a.limb) {
        switch (a.lim) {
        case LIM_VANLEER: return fused_tile<DIR, P, LIM_VANLEER>(a, first, last, st);
        case LIM_MINMOD: return fused_tile<DIR, P, LIM_MINMOD>(a, first, last, st);
        case LIM_MONCEN: return fused_tile<DIR, P, LIM_MONCEN>(a, first, last, st);
        case LIM_SUPERBEE: return fused_tile<DIR, P, LIM_SUPERBEE>(a, first, last, st);
        default: break;
        }
    }
    return fused_tile<DIR, P, -1>(a, first, last, st);
}

template <int DIR, class P, int LIM>
hipError_t flux_tile(const UnsplitArgs &a, double *F, hipStream_t st)
{
    const int d1 = (DIR == 0) ? 1 : 0, d2 = (DIR == 2) ? 1 : 2;
    const long long npen = (long long)a.n[d1] * a.n[d2];
    int TP, TS;
    unsplit_tile<DIR>(a.n[DIR] + 1, npen, 3, TP, TS);
    const int chunks = (a.n[DIR] + 1 + (TS - 3) - 1) / (TS - 3);
    const int nt = (TP * TS + 63) / 64 * 64;
    const long long tiles = (npen + TP - 1) / TP * chunks;
    if (tiles < 1 || tiles > 0x7fffffffll) return hipErrorInvalidValue;
    const size_t shm = sizeof(double) * 2 * P::NV * nt;
    hipLaunchKernelGGL((k_unsplit_flux_tile<DIR, P, LIM>), dim3((unsigned)tiles), dim3(nt), shm, st, a, F, TP,
                       TS, chunks);
    return hipGetLastError();
}

template <int DIR, class P>
hipError_t flux_lim(const UnsplitArgs &a, double *F, unsigned blocks, hipStream_t st)
{
    if (a.lim == a.limb) {
        switch (a.lim) {
        case LIM_VANLEER: return flux_tile<DIR, P, LIM_VANLEER>(a, F, st);
        case LIM_MINMOD: return flux_tile<DIR, P, LIM_MINMOD>(a, F, st);
        case LIM_MONCEN: return flux_tile<DIR, P, LIM_MONCEN>(a, F, st);
        case LIM_SUPERBEE: return flux_tile<DIR, P, LIM_SUPERBEE>(a, F, st);
        default: break;
        }
    }
    return flux_tile<DIR, P, -1>(a, F, st);
}

}  // namespace

hipError_t launch_unsplit_flux(int dir, bool mhd, const UnsplitArgs &a, double *F, hipStream_t st)
{
    if (dir < 0 || dir > 2 || !a.has_dir[dir] || a.g[dir] < 2) return hipErrorInvalidValue;
    const int d1 = (dir == 0) ? 1 : 0, d2 = (dir == 2) ? 1 : 2;
    const long long total = ((long long)a.n[dir] + 1) * a.n[d1] * a.n[d2];
    const long long blocks = (total + 255) / 256;
    if (blocks < 1 || blocks > 0x7fffffffll) return hipErrorInvalidValue;
    if (mhd) {
        if (dir == 0) return flux_lim<0, MHD>(a, F, (unsigned)blocks, st);
        if (dir == 1) return flux_lim<1, MHD>(a, F, (unsigned)blocks, st);
        return flux_lim<2, MHD>(a, F, (unsigned)blocks, st);
    }
    if (dir == 0) return flux_lim<0, HD>(a, F, (unsigned)blocks, st);
    if (dir == 1) return flux_lim<1, HD>(a, F, (unsigned)blocks, st);
    return flux_lim<2, HD>(a, F, (unsigned)blocks, st);
}

hipError_t launch_unsplit_fused(int dir, bool mhd, const UnsplitArgs &a, int first, int last, hipStream_t st)
{
    if (dir < 0 || dir > 2 || !a.has_dir[dir] || a.g[dir] < 2 || a.src == a.dst) return hipErrorInvalidValue;
    if (mhd) {
        if (dir == 0) return fused_lim<0, MHD>(a, first, last, st);
        if (dir == 1) return fused_lim<1, MHD>(a, first, last, st);
        return fused_lim<2, MHD>(a, first, last, st);
    }
    if (dir == 0) return fused_lim<0, HD>(a, first, last, st);
    if (dir == 1) return fused_lim<1, HD>(a, first, last, st);
    return fused_lim<2, HD>(a, first, last, st);
}

hipError_t launch_unsplit_update(bool mhd, const UnsplitArgs &a, const double *const F[3], hipStream_t st)
{
    const long long total = (long long)a.n[0] * a.n[1] * a.n[2];
    const long long blocks = (total + 255) / 256;
    if (blocks < 1 || blocks > 0x7fffffffll) return hipErrorInvalidValue;
    if (mhd)
        hipLaunchKernelGGL(k_unsplit_update<MHD>, dim3((unsigned)blocks), dim3(256), 0, st, a, F[0], F[1], F[2]);
    else
        hipLaunchKernelGGL(k_unsplit_update<HD>, dim3((unsigned)blocks), dim3(256), 0, st, a, F[0], F[1], F[2]);
    return hipGetLastError();
}

}  // namespace PK_KNS
