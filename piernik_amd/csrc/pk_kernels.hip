// pk_kernels.hip -- gfx950 kernels of the split Riemann sweep.
//
// Device layout of one grid block: SoA planes of FP64, one plane per
// variable in xyz order [rho, mx, my, mz, E (, Bx, By, Bz, psi)], each plane
// the ghost-padded box (x fastest):  a[v*sv + x + sy*y + sz*z].
//
// The sweep kernel maps one lane to one cell of a tile of TP pencils x TS
// cells along the sweep direction and exchanges neighbour values (primitive
// states, face states, fluxes) through LDS.  Lanes along x are consecutive,
// so every global load and store is coalesced in all three directions.  In
// FUSED mode both RK2 stages (rk_coef = 1/2, 1; constants.F90:237-238) run in
// one pass: the tile recomputes stage 1 on a 4-cell halo, so U is read once
// and U1 written once; intermediates never leave the CU.  In STAGE mode one
// stage runs over whole pencils exactly as one solve_cg_riemann call does
// (solve_cg_riemann.F90:170-228), pencil ends included.
#include <hip/hip_runtime.h>
#include "pk_math.hpp"
#include "pk_mass.hpp"
#include "pk_kernels.hpp"

namespace PK_KNS {

using pk::ListArgs;
using pk::StepScalars;
using pk::SweepArgs;

#include "pk_tile.hpp"

// Fine/coarse flux points of pencil pf at the right face of cell cs, in
// solve's order (solve_cg_riemann.F90:353-363): a flux sent by a finer
// neighbour replaces the computed one (li, ri), then the flux at a face that
// borders a coarser neighbour is saved (lo, ro), by the one lane that owns
// the cell.  Sweep-order u-fluxes of this fluid, then [B, psi].
template <class P>
__device__ __forceinline__ void fc_points(const SweepArgs &a, int pf, int cs, bool own, double (&F)[P::NV])
{
    const long long np = a.fc_npen;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        if (a.fc_at[k * np + pf] != cs) continue;
        const double *r = a.fc_in + (long long)a.fc_slot[k * np + pf] * a.fc_rec;
#pragma unroll
        for (int v = 0; v < P::NV; v++) F[v] = r[v < 5 ? a.fc_beg + v : a.fc_boff + (v - 5)];
    }
    if (!own) return;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        if (a.fc_at[(2 + k) * np + pf] != cs) continue;
        double *r = a.fc_out + (long long)a.fc_slot[(2 + k) * np + pf] * a.fc_rec;
#pragma unroll
        for (int v = 0; v < P::NV; v++) r[v < 5 ? a.fc_beg + v : a.fc_boff + (v - 5)] = F[v];
    }
}

// One RK stage of the tile.  A holds primitives then fluxes, B face states.
// LIM >= 0 fixes both limiters at compile time; LIM < 0 reads them from a.
// FC: apply the fine/coarse flux points of pencil fc_pf (-1: none) at the
// lane's cell fc_cs; fc_own marks the lane that writes saved fluxes.
template <class P, int LIM, bool FC = false>
__device__ __forceinline__ void tile_stage(const SweepArgs &a, const double (&W)[P::NV],
                                           const double (&W0)[P::NV], double coef, bool upd,
                                           bool lo_end, bool hi_end, double *__restrict__ A,
                                           double *__restrict__ B, int t, int tm, int tp,
                                           double (&Wn)[P::NV], int fc_pf = -1, int fc_cs = 0,
                                           bool fc_own = false)
{
    constexpr int NV = P::NV;
    double fp[NV];
    {
        double q[NV], qm[NV], qp[NV], fm[NV];
        prim<P>(W, a.gam_1, q);
        lds_put<NV>(A, t, q);
        __syncthreads();
        lds_get<NV>(A, tm, qm);
        lds_get<NV>(A, tp, qp);
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const int lim = (LIM >= 0) ? LIM : ((v < 5) ? a.lim : a.limb);
            const double dl = q[v] - qm[v];
            const double dr = qp[v] - q[v];
            double dq;
            if (lo_end)
                dq = (lim == LIM_VANLEER) ? 0.0 : limit(lim, dr, dr);
            else if (hi_end)
                dq = (lim == LIM_VANLEER) ? 0.0 : limit(lim, dl, dl);
            else
                dq = limit(lim, dl, dr);
            const double h = 0.5 * dq;
            fp[v] = q[v] + h;
            fm[v] = q[v] - h;
        }
        lds_put<NV>(B, t, fm);
    }
    __syncthreads();

    double fr[NV], F[NV];
    lds_get<NV>(B, tp, fr);
    if constexpr (P::MAG)
        flux_hlld(fp, fr, a.gam, a.ch, F);
    else
        flux_hllc(fp, fr, a.gam, F);
    if constexpr (FC) {
        if (a.fc_at && fc_pf >= 0) fc_points<P>(a, fc_pf, fc_cs, fc_own, F);
    }
    lds_put<NV>(A, t, F);
    __syncthreads();

    double Fm[NV];
    lds_get<NV>(A, tm, Fm);
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const double un = upd ? W0[v] + coef * (Fm[v] - F[v]) : W[v];
        Wn[v] = (v < 5) ? un + 0.0 : un;  // internal_sources adds +0 to the fluid part
    }
}

// timestep_fluid of the cell a lane has just written (valid lanes), reduced
// over the wave into one slot.
template <int DIR, class P>
__device__ __forceinline__ void dt_contribution(const SweepArgs &a, const double (&Wn)[P::NV], bool valid,
                                                unsigned slot_id)
{
    const double huge = 1.7976931348623157e308;
    double mn[3] = {huge, huge, huge}, cmax = 0.0;
    if (valid) dt_cell<DIR, P>(a, Wn, mn, cmax);
    dt_reduce(a, mn, cmax, slot_id);
}

// One tile of a sweep: chunk `bid % chunks` along the sweep direction times
// TP consecutive pencils of the transverse interior, flattened with d1
// fastest (tile `bid / chunks`).  Lanes t >= TP*TS of a larger workgroup
// take part in the barriers only.  slot_id picks the timestep slot.
template <int DIR, class P, bool FUSED, int LIM>
__device__ __forceinline__ void sweep_tile(const SweepArgs &a, int bid, unsigned slot_id, double *__restrict__ LA,
                                           double *__restrict__ LB)
{
    constexpr int NV = P::NV;
    constexpr int HALO = FUSED ? 4 : 2;
    const int nt = blockDim.x;
    const int t = threadIdx.x;

    constexpr int ds = DIR;
    constexpr int d1 = (DIR == 0) ? 1 : 0;
    constexpr int d2 = (DIR == 2) ? 1 : 2;

    int p, s, tm, tp;
    if (DIR == 0) {
        p = small_div(t, a.TS);
        s = t - p * a.TS;
        tm = t - 1;
        tp = t + 1;
    } else {
        s = small_div(t, a.TP);
        p = t - s * a.TP;
        tm = t - a.TP;
        tp = t + a.TP;
    }
    tm = tm < 0 ? 0 : tm;
    tp = tp >= nt ? nt - 1 : tp;

    const int ptile = a.chunks == 1 ? bid : bid / a.chunks;
    const int chunk = bid - ptile * a.chunks;
    const int n1 = a.n[d1];
    const int npen = n1 * a.n[d2];
    const int pf = ptile * a.TP + p;
    const bool pvalid = t < a.TP * a.TS && pf < npen;
    // transverse coordinates of pencil pf (of the tile's first one, a uniform
    // division, then p further along d1); lanes past the last pencil use it
    int c1, c2;
    if (a.TP <= n1) {
        const int p0 = ptile * a.TP;
        c2 = p0 / n1;
        c1 = p0 - c2 * n1 + p;
        if (c1 >= n1) {
            c1 -= n1;
            c2++;
        }
        if (pf >= npen) {
            c1 = n1 - 1;
            c2 = a.n[d2] - 1;
        }
    } else {
        const int pfc = pf < npen ? pf : npen - 1;
        c2 = pfc / n1;
        c1 = pfc - c2 * n1;
    }
    c1 += a.g[d1];
    c2 += a.g[d2];
    const int ng = a.ng[ds];
    const int os = (FUSED ? a.g[ds] : 0) + chunk * a.out;
    const int oe = FUSED ? a.g[ds] + a.n[ds] : ng;
    const int cs = os - HALO + s;
    const bool svalid = cs >= 0 && cs < ng;
    int csc = cs < 0 ? 0 : (cs >= ng ? ng - 1 : cs);
    if (FUSED && a.wrap) csc = wrap_cell(csc, a.g[ds], a.n[ds]);
    const bool outl = pvalid && s >= HALO && s < HALO + a.out && cs < oe;

    int xyz[3];
    xyz[ds] = csc;
    xyz[d1] = c1;
    xyz[d2] = c2;
    const long long idx = (long long)xyz[0] + (long long)a.sy * xyz[1] + (long long)a.sz * xyz[2];

    double W[NV], W0[NV], Wn[NV];
#pragma unroll
    for (int k = 0; k < NV; k++) W[k] = a.src[(long long)plane_of<DIR>(k) * a.sv + idx];

    // Floor bookkeeping.  Flags: stage 1 over every cell whose stage-1 value
    // the tile completes within two cells of the interior (lanes 2..TS-3;
    // the reference's stage computes these cells with the same stencil), the
    // last stage over the cells the tile writes.  Mass: the interior cells,
    // each stage's events added exactly (pk_mass.hpp).
    unsigned flags = 0u;
    if constexpr (FUSED) {
        double Ws[NV];
        tile_stage<P, LIM>(a, W, W, a.c1, true, false, false, LA, LB, t, tm, tp, Ws);
        double dm = 0.0;
        unsigned fl = 0u;
        floors<P>(Ws, a.smalld, a.smallei, a.use_smalld, a.use_smallei, a.ei_flag, fl, dm);
        const int g = a.g[ds];
        if (pvalid && s >= 2 && s <= a.TS - 3 && cs >= g - 2 && cs < g + a.n[ds] + 2) flags |= fl;
        pk::mass_add(a.dmass, outl ? dm : 0.0);
        tile_stage<P, LIM>(a, Ws, W, a.c2, true, false, false, LB, LA, t, tm, tp, Wn);
    } else {
        const bool lo = cs == 0, hi = cs == ng - 1;
        if (outl && a.base != a.src) {
#pragma unroll
            for (int k = 0; k < NV; k++) W0[k] = a.base[(long long)plane_of<DIR>(k) * a.sv + idx];
        } else {
#pragma unroll
            for (int k = 0; k < NV; k++) W0[k] = W[k];
        }
        tile_stage<P, LIM, true>(a, W, W0, a.c1, !(lo || hi), lo, hi, LA, LB, t, tm, tp, Wn, pvalid ? pf : -1,
                                 cs, outl && svalid);
    }
    {
        double dm = 0.0;
        unsigned fl = 0u;
        floors<P>(Wn, a.smalld, a.smallei, a.use_smalld, a.use_smallei, a.ei_flag, fl, dm);
        const bool inner = cs >= a.g[ds] && cs < a.g[ds] + a.n[ds];
        if (outl) flags |= fl;
        pk::mass_add(a.dmass, (outl && inner) ? dm : 0.0);
    }
    if constexpr (FUSED) {
        if (a.dtslots) dt_contribution<DIR, P>(a, Wn, outl && svalid, slot_id);
    }
    if constexpr (P::MAG) Wn[8] = Wn[8] * a.psi_fac;

    if (outl && svalid) {
#pragma unroll
        for (int k = 0; k < NV; k++) a.dst[(long long)plane_of<DIR>(k) * a.sv + idx] = Wn[k];
    }
    // negative values are rare: one atomic per lane that saw one
    if (flags) atomicOr(a.flags, flags);
}

// ---------------------------------------------------------------- march ----
// The fused RK2 sweep with one lane per pencil.  A lane walks its pencil
// cell by cell and carries a register window instead of sharing neighbours
// through LDS: the primitives of the last two cells and the last face state
// and flux of each stage.  Reading cell t it completes the stage-1 flux at
// (t-2)+1/2, the stage-1 state of cell t-2, the stage-2 flux at (t-4)+1/2 and
// the new state of cell t-4.  No cell is computed twice, no barrier is needed,
// and for y and z sweeps consecutive lanes are consecutive x, so every load
// and store is coalesced.  Each cell sees the operands and operations of the
// tile kernel in the same order: the results are bit-identical.

template <class P, int LIM>
__device__ __forceinline__ void cell_faces(const SweepArgs &a, const double (&qm)[P::NV], const double (&q)[P::NV],
                                           const double (&qp)[P::NV], double (&fp)[P::NV], double (&fm)[P::NV])
{
#pragma unroll
    for (int v = 0; v < P::NV; v++) {
        const int lim = (LIM >= 0) ? LIM : ((v < 5) ? a.lim : a.limb);
        const double dl = q[v] - qm[v];
        const double dr = qp[v] - q[v];
        const double h = 0.5 * limit(lim, dl, dr);
        fp[v] = q[v] + h;
        fm[v] = q[v] - h;
    }
}

template <class P>
__device__ __forceinline__ void riemann(const SweepArgs &a, const double (&l)[P::NV], const double (&r)[P::NV],
                                        double (&F)[P::NV])
{
    if constexpr (P::MAG)
        flux_hlld(l, r, a.gam, a.ch, F);
    else
        flux_hllc(l, r, a.gam, F);
}

template <class P>
__device__ __forceinline__ void cell_update(const double (&W0)[P::NV], double coef, const double (&Fm)[P::NV],
                                            const double (&Fp)[P::NV], double (&Wn)[P::NV])
{
#pragma unroll
    for (int v = 0; v < P::NV; v++) {
        const double un = W0[v] + coef * (Fm[v] - Fp[v]);
        Wn[v] = (v < 5) ? un + 0.0 : un;  // internal_sources adds +0 to the fluid part
    }
}

template <int NV>
__device__ __forceinline__ void copy_nv(double (&d)[NV], const double (&s)[NV])
{
#pragma unroll
    for (int v = 0; v < NV; v++) d[v] = s[v];
}

template <int DIR, class P, int LIM>
__global__ __launch_bounds__(64) void k_march(const SweepArgs a)
{
    constexpr int NV = P::NV;
    constexpr int ds = DIR;
    constexpr int d1 = (DIR == 0) ? 1 : 0;
    constexpr int d2 = (DIR == 2) ? 1 : 2;
    const int n1 = a.n[d1];
    const int npen = n1 * a.n[d2];
    const int pf = blockIdx.x * blockDim.x + threadIdx.x;
    const bool pvalid = pf < npen;
    const int pfc = pvalid ? pf : npen - 1;
    int xyz[3];
    xyz[d1] = a.g[d1] + pfc % n1;
    xyz[d2] = a.g[d2] + pfc / n1;
    xyz[ds] = 0;
    const long long step = (DIR == 0) ? 1ll : ((DIR == 1) ? (long long)a.sy : (long long)a.sz);
    const long long base = (long long)xyz[0] + (long long)a.sy * xyz[1] + (long long)a.sz * xyz[2];
    const int g = a.g[ds], n = a.n[ds];
    const int t0 = g - 4, t1 = g + n + 4;  // cells read: [t0, t1)

    auto load = [&](int c, double (&W)[NV]) {
        c = c < t0 ? t0 : (c >= t1 ? t1 - 1 : c);
        if (a.wrap) c = wrap_cell(c, g, n);
        const long long o = base + step * c;
#pragma unroll
        for (int k = 0; k < NV; k++) W[k] = a.src[(long long)plane_of<DIR>(k) * a.sv + o];
    };

    // the window (values before the pipeline fills are never stored)
    double qa[NV], qb[NV];    // primitives of cells t-2, t-1
    double fpp[NV], F1m[NV];  // stage 1: face state on the right of cell t-2; flux at (t-2)-1/2
    double sa[NV], sb[NV];    // stage-1 primitives of cells t-4, t-3
    double fps[NV], F2m[NV];  // stage 2: face state on the right of cell t-4; flux at (t-4)-1/2
#pragma unroll
    for (int v = 0; v < NV; v++) qa[v] = qb[v] = fpp[v] = F1m[v] = sa[v] = sb[v] = fps[v] = F2m[v] = 1.0;

    unsigned flags = 0u;
    const double huge = 1.7976931348623157e308;
    double mn[3] = {huge, huge, huge}, cmax = 0.0;
    double Wnext[NV];
    load(t0, Wnext);
    for (int t = t0; t < t1; t++) {
        double W[NV], W2[NV], W4[NV];
        copy_nv(W, Wnext);
        load(t + 1, Wnext);
        load(t - 2, W2);
        load(t - 4, W4);
        double q[NV];
        prim<P>(W, a.gam_1, q);
        // stage 1: face states of cell t-1, flux at (t-2)+1/2, state of cell t-2
        double fp[NV], fm[NV], F1[NV];
        cell_faces<P, LIM>(a, qa, qb, q, fp, fm);
        riemann<P>(a, fpp, fm, F1);
        double Ws[NV];
        cell_update<P>(W2, a.c1, F1m, F1, Ws);
        {
            // the stage-1 value of cell t-2 is complete from t = g on (cells
            // from g-2: the two cells next to the interior, as the tiles)
            unsigned fl = 0u;
            double dm = 0.0;
            floors<P>(Ws, a.smalld, a.smallei, a.use_smalld, a.use_smallei, a.ei_flag, fl, dm);
            const int c = t - 2;
            if (c >= g - 2) flags |= fl;
            pk::mass_add(a.dmass, (pvalid && c >= g && c < g + n) ? dm : 0.0);
        }
        double qs[NV];
        prim<P>(Ws, a.gam_1, qs);
        // stage 2: face states of cell t-3, flux at (t-4)+1/2, new state of cell t-4
        double gp[NV], gm[NV], F2[NV];
        cell_faces<P, LIM>(a, sa, sb, qs, gp, gm);
        riemann<P>(a, fps, gm, F2);
        double Wn[NV];
        cell_update<P>(W4, a.c2, F2m, F2, Wn);
        const int c = t - 4;
        {
            unsigned fl = 0u;
            double dm = 0.0;
            floors<P>(Wn, a.smalld, a.smallei, a.use_smalld, a.use_smallei, a.ei_flag, fl, dm);
            if (c >= g) flags |= fl;
            pk::mass_add(a.dmass, (pvalid && c >= g) ? dm : 0.0);
        }
        if (c >= g) {
            if (a.dtslots && pvalid) dt_cell<DIR, P>(a, Wn, mn, cmax);
            if constexpr (P::MAG) Wn[8] = Wn[8] * a.psi_fac;
            if (pvalid) {
                const long long idx = base + step * c;
#pragma unroll
                for (int k = 0; k < NV; k++) a.dst[(long long)plane_of<DIR>(k) * a.sv + idx] = Wn[k];
            }
        }
        // advance the window
        copy_nv(qa, qb);
        copy_nv(qb, q);
        copy_nv(fpp, fp);
        copy_nv(F1m, F1);
        copy_nv(sa, sb);
        copy_nv(sb, qs);
        copy_nv(fps, gp);
        copy_nv(F2m, F2);
    }
    if (a.dtslots) dt_reduce(a, mn, cmax, blockIdx.x);
    if (pvalid && flags) atomicOr(a.flags, flags);
}

// The kernel arguments of list item `item` (its block's table entry with
// the step's scalars and buffer parity applied); returns the block's first
// item, and in `next` the first item past it.  The tables are read-only while a kernel runs: they are read through
// the constant address space, so the uniform loads go to scalar registers.
template <int DIR>
__device__ __forceinline__ unsigned load_list_args(const ListArgs &L, unsigned item, SweepArgs &a, unsigned &next)
{
    typedef const __attribute__((address_space(4))) unsigned cu32;
    const int blk = __builtin_amdgcn_readfirstlane((int)((cu32 *)L.items)[item]);
    {
        static_assert(sizeof(SweepArgs) % 4 == 0, "SweepArgs is copied in dwords");
        cu32 *w = (cu32 *)(L.args + blk);
        unsigned *aw = reinterpret_cast<unsigned *>(&a);
#pragma unroll
        for (int i = 0; i < (int)(sizeof(SweepArgs) / 4); i++) aw[i] = w[i];
    }
    const unsigned first = ((cu32 *)L.first)[blk];
    next = ((cu32 *)L.first)[blk + 1];
    if (L.given) a.wrap = 0;
    if (L.parity) {
        const double *s0 = a.src;
        a.src = a.dst;
        a.dst = const_cast<double *>(s0);
    }
    a.base = a.src;
    typedef const __attribute__((address_space(4))) double cf64;
    const int inst = L.per_block ? (L.bpos ? (int)((cu32 *)L.bpos)[blk] : blk) : 0;
    const cf64 *stp = (const cf64 *)(L.step + inst);
    const double sdt = stp[0], sch = stp[1], sfac = stp[2];
    a.c1 = (0.5 * sdt) / a.dl[DIR];  // rk_coef * dt / dl, constants.F90:237-238
    a.c2 = (1.0 * sdt) / a.dl[DIR];
    a.ch = sch;
    a.psi_fac = L.apply_fac ? sfac : 1.0;
    a.dtslots = L.dtslots ? L.dtslots + 4ll * L.nslots * inst : nullptr;
    a.nslots = L.nslots;
    return first;
}

#include "pk_stream.hpp"

// Hydro tiles hold five waves per SIMD (86 VGPRs), fused MHD tiles are held to
// three (168 VGPRs, 8-10 of them spilled; unconstrained 175-185, two waves):
// four steps of a 131x98x77 MHD block took 4020 us with two, 3770 with three.
// The one-stage MHD sweep would spill 24 and keeps two (100 against 90 us).
template <int DIR, class P, bool FUSED, int LIM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(P::MAG ? (FUSED ? 3 : 2) : 5))) void k_sweep(const SweepArgs a)
{
    extern __shared__ double lds[];
    unsigned bid = pk::xcd_order();
    if constexpr (!FUSED) {
        // A stage writes transverse-interior pencils; the other cells of dst
        // take src's values, as the reference leaves them, from workgroups of
        // the same launch (96^3 MHD: a launch of its own over every cell took
        // 10.6 us after each 67 us stage, this adds 7 us).
        if (blockIdx.x < (unsigned)a.gwgs) {
            unsigned n[3], g[3], c[3];
#pragma unroll
            for (int d = 0; d < 3; d++) {
                n[d] = (unsigned)(d == DIR ? a.ng[d] : a.n[d]);
                g[d] = (unsigned)(d == DIR ? 0 : a.g[d]);
            }
            if (pk::ghost_cell(blockIdx.x * blockDim.x + threadIdx.x, n, g, c)) {
                const long long i = c[0] + (long long)a.sy * c[1] + (long long)a.sz * c[2];
                pk::copy_planes<P::NV>(a.src + i, a.sv, a.dst + i, a.sv, P::NV);
            }
            return;
        }
        bid = pk::xcd_order(blockIdx.x - (unsigned)a.gwgs, gridDim.x - (unsigned)a.gwgs);
    }
    sweep_tile<DIR, P, FUSED, LIM>(a, (int)bid, blockIdx.x, lds, lds + P::NV * blockDim.x);
}

// Fused sweep over a block list, a tile per workgroup.
template <int DIR, class P, int LIM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(P::MAG ? 3 : 5))) void k_sweep_list(const ListArgs L)
{
    extern __shared__ double lds[];
    const unsigned item = L.item0 + pk::xcd_order();
    SweepArgs a;
    unsigned next;
    const unsigned first = load_list_args<DIR>(L, item, a, next);
    sweep_tile<DIR, P, true, LIM>(a, (int)(item - first), item, lds, lds + P::NV * blockDim.x);
}

// ------------------------------------------------------------ launchers ----

template <int DIR, class P, bool FUSED, int LIM>
static hipError_t launch_sweep_t(const SweepArgs &a, hipStream_t st)
{
    const int nt = a.TP * a.TS;
    const size_t lds = sizeof(double) * 2 * P::NV * nt;
    static bool lds_raised = false;  // allow dynamic LDS beyond 64 KiB (gfx950 has 160 KiB per CU)
    if (!lds_raised) {
        hipError_t e = hipFuncSetAttribute((const void *)k_sweep<DIR, P, FUSED, LIM>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        lds_raised = true;
    }
    if (lds > 160 * 1024 || nt > 512) return hipErrorInvalidValue;
    const long long nblk = (long long)a.chunks * a.ptiles;
    if constexpr (FUSED) {
        hipLaunchKernelGGL((k_sweep<DIR, P, FUSED, LIM>), dim3((unsigned)nblk), dim3(nt), lds, st, a);
    } else {
        const int d1 = (DIR == 0) ? 1 : 0, d2 = (DIR == 2) ? 1 : 2;
        const long long cells = ((long long)a.ng[d1] * a.ng[d2] - (long long)a.n[d1] * a.n[d2]) * a.ng[DIR];
        if (cells > 0xffff0000ll) return hipErrorInvalidValue;  // more cells than memory holds
        SweepArgs s = a;
        s.gwgs = (int)(((cells + nt - 1) / nt + 7) / 8 * 8);
        hipLaunchKernelGGL((k_sweep<DIR, P, FUSED, LIM>), dim3((unsigned)(nblk + s.gwgs)), dim3(nt), lds, st, s);
    }
    return hipGetLastError();
}

template <int DIR, class P, int LIM>
static hipError_t launch_march_t(const SweepArgs &a, hipStream_t st)
{
    const int d1 = (DIR == 0) ? 1 : 0, d2 = (DIR == 2) ? 1 : 2;
    const long long npen = (long long)a.n[d1] * a.n[d2];
    const long long nblk = (npen + 63) / 64;
    if (a.g[DIR] < 4 || nblk < 1 || nblk > 0x7fffffffll) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_march<DIR, P, LIM>), dim3((unsigned)nblk), dim3(64), 0, st, a);
    return hipGetLastError();
}

constexpr int kMaxDevices = 64;

// Workgroups of `fn` (one wave each) resident on the current device at
// once, 0 if unknown; cached per device.
static int stream_slots(const void *fn, int *cache)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
    if (cache[dev] == 0) {
        int per = 0, ncu = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, 64, 0) != hipSuccess ||
            hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
            (void)hipGetLastError();  // launch without rounding; leave no error for the launch check
            return 0;
        }
        cache[dev] = per * ncu;
    }
    return cache[dev];
}

// The stream kernel: a.TP pencils per lane group, a.ptiles ranges of whole
// pencil groups (a.out positions each, the last one shorter) asked for.  A
// launch of more ranges than the device holds at once runs in rounds; it is
// rounded to a whole number of rounds, the ranges made equal to within one
// group, so that the last round does not leave the device partly idle.
template <int DIR, class P, int LIM, int TP>
static hipError_t launch_stream_tp(const SweepArgs &a, hipStream_t st)
{
    constexpr int d1 = (DIR == 0) ? 1 : 0, d2 = (DIR == 2) ? 1 : 2;
    const long long npen = (long long)a.n[d1] * a.n[d2];
    const long long L = a.n[DIR] + 8;
    const long long ngroups = (npen + TP - 1) / TP;
    const long long npos = ngroups * L;
    const int span = a.out;
    if (a.g[DIR] < 4 || span <= 0 || span % L != 0 || npos + span + 64 > 0x7fffffffll || !pk::stream_stores_fit(a.sv))
        return hipErrorInvalidValue;
    long long nblk = (npos + span - 1) / span;
    if (nblk != a.ptiles) return hipErrorInvalidValue;
    const void *fn = (const void *)k_stream<DIR, P, LIM, TP>;
    static int cache[kMaxDevices] = {};
    const long long slots = stream_slots(fn, cache);
    if (slots > 0 && nblk >= slots) {
        // nblk <= ngroups, so one round of slots ranges has a group each
        long long r = (nblk + slots / 2) / slots;
        while (r > 1 && r * slots > ngroups) r--;
        nblk = r * slots;
    }
    hipLaunchKernelGGL((k_stream<DIR, P, LIM, TP>), dim3((unsigned)nblk), dim3(64), 0, st, a, (int)ngroups);
    return hipGetLastError();
}

template <int DIR, class P, int LIM>
static hipError_t launch_stream_t(const SweepArgs &a, hipStream_t st)
{
    switch (a.TP) {
    case 1: return launch_stream_tp<DIR, P, LIM, 1>(a, st);
    case 2: return launch_stream_tp<DIR, P, LIM, 2>(a, st);
    case 4: return launch_stream_tp<DIR, P, LIM, 4>(a, st);
    case 8: return launch_stream_tp<DIR, P, LIM, 8>(a, st);
    default: return hipErrorInvalidValue;
    }
}

template <int DIR, class P, bool FUSED>
static hipError_t launch_lim(const SweepArgs &a, hipStream_t st)
{
    if constexpr (FUSED) {
        if (a.TS <= -2) {  // the stream kernel (k_stream)
            if (a.lim == a.limb) {
                switch (a.lim) {
                case LIM_VANLEER: return launch_stream_t<DIR, P, LIM_VANLEER>(a, st);
                case LIM_MINMOD: return launch_stream_t<DIR, P, LIM_MINMOD>(a, st);
                case LIM_MONCEN: return launch_stream_t<DIR, P, LIM_MONCEN>(a, st);
                case LIM_SUPERBEE: return launch_stream_t<DIR, P, LIM_SUPERBEE>(a, st);
                default: break;
                }
            }
            return launch_stream_t<DIR, P, -1>(a, st);
        }
        if (a.TS < 0) {  // whole pencils, one lane each (k_march)
            if (a.lim == a.limb) {
                switch (a.lim) {
                case LIM_VANLEER: return launch_march_t<DIR, P, LIM_VANLEER>(a, st);
                case LIM_MINMOD: return launch_march_t<DIR, P, LIM_MINMOD>(a, st);
                case LIM_MONCEN: return launch_march_t<DIR, P, LIM_MONCEN>(a, st);
                case LIM_SUPERBEE: return launch_march_t<DIR, P, LIM_SUPERBEE>(a, st);
                default: break;
                }
            }
            return launch_march_t<DIR, P, -1>(a, st);
        }
    }
    if (a.lim == a.limb) {
        switch (a.lim) {
        case LIM_VANLEER: return launch_sweep_t<DIR, P, FUSED, LIM_VANLEER>(a, st);
        case LIM_MINMOD: return launch_sweep_t<DIR, P, FUSED, LIM_MINMOD>(a, st);
        case LIM_MONCEN: return launch_sweep_t<DIR, P, FUSED, LIM_MONCEN>(a, st);
        case LIM_SUPERBEE: return launch_sweep_t<DIR, P, FUSED, LIM_SUPERBEE>(a, st);
        default: break;
        }
    }
    return launch_sweep_t<DIR, P, FUSED, -1>(a, st);
}

hipError_t launch_sweep(int dir, bool mhd, bool fused, const SweepArgs &a, hipStream_t st)
{
#define PK_CASE(D, PP, F) \
    if (dir == D && (mhd == PP::MAG) && fused == F) return launch_lim<D, PP, F>(a, st);
    PK_CASE(0, HD, true) PK_CASE(1, HD, true) PK_CASE(2, HD, true)
    PK_CASE(0, HD, false) PK_CASE(1, HD, false) PK_CASE(2, HD, false)
    PK_CASE(0, MHD, true) PK_CASE(1, MHD, true) PK_CASE(2, MHD, true)
    PK_CASE(0, MHD, false) PK_CASE(1, MHD, false) PK_CASE(2, MHD, false)
#undef PK_CASE
    return hipErrorInvalidValue;
}

// List sweep: launch (resident == nullptr) or report how many workgroups of nt
// lanes the device holds at once.  nt == 64: the stream (k_stream_list, one
// pencil per lane group along x, eight along y and z).
template <int DIR, class P, int LIM>
static hipError_t stream_list_t(const ListArgs *L, int grid, hipStream_t st, int *resident)
{
    constexpr int TP = pk::stream_list_tp(DIR);
    const void *fn = (const void *)k_stream_list<DIR, P, LIM, TP>;
    if (resident) {
        int per = 0, dev = 0, ncu = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, 64, 0);
        if (e == hipSuccess) e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
        *resident = per * ncu;
        return e;
    }
    if (grid <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_stream_list<DIR, P, LIM, TP>), dim3((unsigned)grid), dim3(64), 0, st, *L);
    return hipGetLastError();
}

template <int DIR, class P, int LIM>
static hipError_t list_t(const ListArgs *L, int nt, int grid, hipStream_t st, int *resident)
{
    if (nt == pk::kStreamListNt) return stream_list_t<DIR, P, LIM>(L, grid, st, resident);
    const void *fn = (const void *)k_sweep_list<DIR, P, LIM>;
    const size_t lds = sizeof(double) * 2 * P::NV * nt;
    const size_t lds_max = 160 * 1024;
    static bool lds_raised = false;
    if (!lds_raised) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max);
        if (e != hipSuccess) return e;
        lds_raised = true;
    }
    if (nt < 64 || nt > 512 || nt % 64 != 0 || lds > lds_max) return hipErrorInvalidValue;
    if (resident) {
        int per = 0, dev = 0, ncu = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, nt, lds);
        if (e == hipSuccess) e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
        *resident = per * ncu;
        return e;
    }
    ListArgs l = *L;
    for (; l.item0 < L->nitems; l.item0 += pk::kListPiece) {
        const unsigned n = L->nitems - l.item0 < pk::kListPiece ? L->nitems - l.item0 : pk::kListPiece;
        hipLaunchKernelGGL((k_sweep_list<DIR, P, LIM>), dim3(n), dim3(nt), lds, st, l);
        if (l.item0 + n == L->nitems) break;  // (the next item0 may not fit 32 bits)
    }
    return hipGetLastError();
}

template <int DIR, class P>
static hipError_t list_lim(int lim, int limb, const ListArgs *L, int nt, int grid, hipStream_t st, int *resident)
{
    if (lim == limb) {
        switch (lim) {
        case LIM_VANLEER: return list_t<DIR, P, LIM_VANLEER>(L, nt, grid, st, resident);
        case LIM_MINMOD: return list_t<DIR, P, LIM_MINMOD>(L, nt, grid, st, resident);
        case LIM_MONCEN: return list_t<DIR, P, LIM_MONCEN>(L, nt, grid, st, resident);
        case LIM_SUPERBEE: return list_t<DIR, P, LIM_SUPERBEE>(L, nt, grid, st, resident);
        default: break;
        }
    }
    return list_t<DIR, P, -1>(L, nt, grid, st, resident);
}

static hipError_t list_dispatch(int dir, bool mhd, int lim, int limb, const ListArgs *L, int nt, int grid,
                                hipStream_t st, int *resident)
{
    if (mhd) {
        if (dir == 0) return list_lim<0, MHD>(lim, limb, L, nt, grid, st, resident);
        if (dir == 1) return list_lim<1, MHD>(lim, limb, L, nt, grid, st, resident);
        if (dir == 2) return list_lim<2, MHD>(lim, limb, L, nt, grid, st, resident);
    } else {
        if (dir == 0) return list_lim<0, HD>(lim, limb, L, nt, grid, st, resident);
        if (dir == 1) return list_lim<1, HD>(lim, limb, L, nt, grid, st, resident);
        if (dir == 2) return list_lim<2, HD>(lim, limb, L, nt, grid, st, resident);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_sweep_list(int dir, bool mhd, int lim, int limb, const ListArgs &L, int nt, int grid,
                             hipStream_t st)
{
    if (nt == pk::kStreamListNt && grid <= 0) {
        int r = 0;
        hipError_t e = list_dispatch(dir, mhd, lim, limb, &L, nt, 0, st, &r);
        if (e != hipSuccess) return e;
        grid = r > 0 ? r : 1;
        if (L.nitems < (unsigned)grid) grid = L.nitems > 0 ? (int)L.nitems : 1;
    }
    return list_dispatch(dir, mhd, lim, limb, &L, nt, grid, st, nullptr);
}

int sweep_list_resident(int dir, bool mhd, int lim, int limb, int nt)
{
    int r = 0;
    if (list_dispatch(dir, mhd, lim, limb, nullptr, nt, 0, nullptr, &r) != hipSuccess) return 0;
    return r;
}

}  // namespace PK_KNS
