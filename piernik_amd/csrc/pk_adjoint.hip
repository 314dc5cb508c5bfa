// pk_adjoint.hip -- reverse mode of the fused RK2 sweep, hydro and MHD (gfx950).
//
// For one directional sweep of a periodic block with hydro fluids
//   U* = floors(U + c1 R(U)),  U' = floors(U + c2 R(U*)),
//   R(W)_i = F(W)_{i-1/2} - F(W)_{i+1/2},  c1 = (dt/2)/dl,  c2 = dt/dl,
// (solve_cg_riemann.F90:366 inside the RK2 loop of sweeps.F90:217-272), the
// kernel takes lam' = dL/dU' and returns lam = dL/dU, plus dL/d(dt), with
// F = HLLC of the limited piecewise-linear face states (hlld.F90:615-841,
// interpolations.F90:112-204).
//
// One lane is one cell of a tile of TP pencils x TS cells along the sweep.
// The tile first recomputes both stages from U (forward values are the
// forward sweep's bit for bit: same functions, same order, no contraction),
// then runs the chain rule backwards; neighbour terms go through LDS.  The
// output cells are lanes 8 .. TS-9: eight cells of halo on each side.
// Reads wrap periodically along the sweep, so ghost cells are not used.
#include <hip/hip_runtime.h>
// the arithmetic of pk_math.hpp and pk_adjoint.hpp without range scaling in
// divisions and square roots, in a namespace of its own
#define PK_KNS pk_adj
#define PK_NORMAL_RANGE 1
#include "pk_adjoint.hpp"
#include "pk_adjoint_kernels.hpp"

namespace pk {

using namespace pk_adj;

template <int DIR>
__device__ __forceinline__ int plane_of_adj(int k)
{
    // sweep-order variable k -> xyz plane (fluidtypes.F90:318-320, fluidindex.F90:190-192)
    if (DIR == 0) return k;
    if (DIR == 1) {
        constexpr int p[9] = {0, 2, 1, 3, 4, 6, 5, 7, 8};
        return p[k];
    }
    constexpr int p[9] = {0, 3, 2, 1, 4, 7, 6, 5, 8};
    return p[k];
}

// limiter of variable v: fluid variables use 'limiter', B and psi 'limiter_b'
template <int LIM>
__device__ __forceinline__ int lim_of(const AdjArgs &a, int v)
{
    return (LIM >= 0) ? LIM : ((v < 5) ? a.lim : a.limb);
}

// limited face states of cell k from q_{k-1}, q_k, q_{k+1}
template <class P, int LIM>
__device__ __forceinline__ void faces(const AdjArgs &a, const double (&qm)[P::NV], const double (&q)[P::NV],
                                      const double (&qp)[P::NV], double (&fp)[P::NV], double (&fm)[P::NV])
{
#pragma unroll
    for (int v = 0; v < P::NV; v++) {
        const double dq = limit(lim_of<LIM>(a, v), q[v] - qm[v], qp[v] - q[v]);
        const double h = 0.5 * dq;
        fp[v] = q[v] + h;
        fm[v] = q[v] - h;
    }
}

// One lane's NV values of an LDS array, lane by lane (NV is odd: consecutive
// lanes fall on different banks): one address per array and lane, the
// variables at immediate offsets.  With the variables nt apart, nt a run-time
// value, the MHD kernel held an address register per variable and array and
// spilled them (395 scratch accesses in its code).
template <int NV>
__device__ __forceinline__ void lds_get(const double *A, int t, double (&x)[NV])
{
#pragma unroll
    for (int v = 0; v < NV; v++) x[v] = A[t * NV + v];
}
template <int NV>
__device__ __forceinline__ void lds_put(double *A, int t, const double (&x)[NV])
{
#pragma unroll
    for (int v = 0; v < NV; v++) A[t * NV + v] = x[v];
}

// LDS arrays of NV doubles per lane of the adjoint tile.
constexpr int kAdjArrays = 4;

// q_bar of cell k from its face-state adjoints (fpb: left state of k+1/2,
// fmb: right state of k-1/2) through the limiter: the own-cell part and the
// dl/dr adjoints that the neighbours take.
template <class P, int LIM>
__device__ __forceinline__ void faces_vjp(const AdjArgs &a, const double (&qm)[P::NV], const double (&q)[P::NV],
                                          const double (&qp)[P::NV], const double (&fpb)[P::NV],
                                          const double (&fmb)[P::NV], double (&qb)[P::NV], double (&dlb)[P::NV],
                                          double (&drb)[P::NV])
{
#pragma unroll
    for (int v = 0; v < P::NV; v++) {
        const double dqb = 0.5 * fpb[v] - 0.5 * fmb[v];
        limit_vjp(lim_of<LIM>(a, v), q[v] - qm[v], qp[v] - q[v], dqb, dlb[v], drb[v]);
        qb[v] = (fpb[v] + fmb[v]) + (dlb[v] - drb[v]);
    }
}

template <class P>
__device__ __forceinline__ void flux(const AdjArgs &a, const double *l, const double *r, double *F)
{
    if constexpr (P::MAG)
        flux_hlld(l, r, a.gam, a.ch, F);
    else
        flux_hllc(l, r, a.gam, F);
}

// returns dL/dch of this interface
template <class P>
__device__ __forceinline__ double flux_vjp(const AdjArgs &a, const double *l, const double *r, const double *fb,
                                           double *lb, double *rb)
{
    if constexpr (P::MAG) {
        return hlld_vjp_r(l, r, a.gam, a.rg, a.rg1, a.ch, a.rch, fb, lb, rb);
    } else {
        hllc_vjp_r(l, r, a.gam, a.rg1, fb, lb, rb);
        return 0.0;
    }
}

template <class P>
__device__ __forceinline__ void floors_vjp(const AdjArgs &a, const double (&u)[P::NV], double (&ub)[P::NV])
{
    if constexpr (P::MAG)
        floors_vjp_mhd(u, a.smalld, a.smallei, a.use_smalld, a.use_smallei, ub);
    else
        floors_vjp_hd(u, a.smalld, a.smallei, a.use_smalld, a.use_smallei, ub);
}

template <class P>
__device__ __forceinline__ void prim_vjp(const AdjArgs &a, const double (&u)[P::NV], const double (&qb)[P::NV],
                                         double (&ub)[P::NV])
{
    if constexpr (P::MAG)
        prim_vjp_mhd(u, a.gam_1, qb, ub);
    else
        prim_vjp_hd(u, a.gam_1, qb, ub);
}

// One tile (bid) of the adjoint sweep; lanes t >= TP*TS of a larger
// workgroup take part in the barriers only.
//
// The tile keeps four LDS arrays of NV doubles per lane (73.7 KB for MHD, so
// that two workgroups, two waves per SIMD, share a CU):
//   Q  primitives of the stage in hand, and once those are used an exchange
//   S  right-face states, then lam' (from the reverse of stage 2 on, own cell)
//   T  fluxes and other neighbour exchanges
//   K  R1 of the own cell until the reverse of stage 1, then exchanges
// An array is rewritten only after a barrier that follows its last read by
// another lane.  U and the stage-1 primitives are formed again where they are
// needed instead of being held across the flux VJPs.
//
// Bound by FP64 VALU issue (hydro: four waves per SIMD, the VALU 86 - 90 %
// busy at 128^3) and, for MHD, by waits (two waves per SIMD, the VALU 41 - 48 %
// busy, half the waves' cycles at s_waitcnt for LDS and scratch).
// Against both-sided flux VJPs with IEEE divisions, eight (hydro five) arrays
// and tiles in launch order: VALU instructions per wave 3143 -> 2136 (hydro)
// and 9508 -> 5000 (MHD), waves per SIMD 2 -> 4 and 1 -> 2; the list sweeps of
// 20 Orszag-Tang instances (64^2 .. 256^2) 527 and 633 us -> 297 and 325 us
// (x, y), a 96^3 hydro rollout with its gradient 7.18 -> 5.3-5.8 ms.  (The
// special values of division cost 1.5 % of a gradient since.)  The
// XCD-aware order is worth 1.4x of that rollout: in launch order the tiles of
// one cache line of a y or z sweep ran on eight L2s (110e6 busy CU cycles per
// y sweep against 49e6 along x; in XCD order 50e6).
template <int DIR, class P, int LIM>
__device__ __forceinline__ void adjoint_tile(const AdjArgs &a, int bid, double *lds)
{
    constexpr int NV = P::NV;
    const int nt = blockDim.x;
    const int t = threadIdx.x;
    double *Q = lds, *S = lds + NV * nt, *T = lds + 2 * NV * nt, *K = lds + 3 * NV * nt;

    constexpr int d1 = (DIR == 0) ? 1 : 0;
    constexpr int d2 = (DIR == 2) ? 1 : 2;
    const int step = (DIR == 0) ? 1 : a.TP;
    int p, s;
    if (DIR == 0) {
        s = t % a.TS;
        p = t / a.TS;
    } else {
        p = t % a.TP;
        s = t / a.TP;
    }
    const int tm = max(t - step, 0), tp = min(t + step, nt - 1);

    const int chunk = bid % a.chunks;
    const int ptile = bid / a.chunks;
    const int n1 = a.n[d1], nd = a.n[DIR];
    const int npen = n1 * a.n[d2];
    const int pf = ptile * a.TP + p;
    const bool pvalid = t < a.TP * a.TS && pf < npen;
    const int pfc = pf < npen ? pf : npen - 1;
    const int c1i = a.g[d1] + pfc % n1;
    const int c2i = a.g[d2] + pfc / n1;
    const int cs = chunk * a.out - 8 + s;  // interior coordinate along the sweep, before wrapping
    const int ci = ((cs % nd) + nd) % nd;
    const bool outl = pvalid && s >= 8 && s < 8 + a.out && cs < nd;

    int xyz[3];
    xyz[DIR] = a.g[DIR] + ci;
    xyz[d1] = c1i;
    xyz[d2] = c2i;
    const long long idx = (long long)xyz[0] + (long long)a.sy * xyz[1] + (long long)a.sz * xyz[2];

    auto load_u = [&](double (&U)[NV]) {
#pragma unroll
        for (int k = 0; k < NV; k++) U[k] = a.u[(long long)plane_of_adj<DIR>(k) * a.sv + idx];
    };
    // the stage-1 state before the floors, from U and R1
    auto stage1 = [&](const double (&U)[NV], const double (&R1)[NV], double (&W)[NV]) {
#pragma unroll
        for (int v = 0; v < NV; v++) {
            const double un = U[v] + a.c1 * R1[v];
            W[v] = (v < 5) ? un + 0.0 : un;
        }
    };
    auto floored = [&](double (&W)[NV]) {
        unsigned fl = 0u;
        double dm = 0.0;
        floors<P>(W, a.smalld, a.smallei, a.use_smalld, a.use_smallei, false, fl, dm);
    };

    double fp[NV], r[NV], F[NV];
    // ---- forward: stage 1 ----
    {
        double U[NV], q[NV], qm[NV], qp[NV], fm[NV];
        load_u(U);
        prim<P>(U, a.gam_1, q);
        lds_put<NV>(Q, t, q);
        __syncthreads();
        lds_get<NV>(Q, tm, qm);
        lds_get<NV>(Q, tp, qp);
        faces<P, LIM>(a, qm, q, qp, fp, fm);
        lds_put<NV>(S, t, fm);
        __syncthreads();
        lds_get<NV>(S, tp, r);
        flux<P>(a, fp, r, F);
        lds_put<NV>(T, t, F);
        __syncthreads();
        double Fm[NV], R1[NV], Us[NV];
        lds_get<NV>(T, tm, Fm);
#pragma unroll
        for (int v = 0; v < NV; v++) R1[v] = Fm[v] - F[v];
        stage1(U, R1, Us);
        floored(Us);
        lds_put<NV>(K, t, R1);
        // ---- forward: stage 2 ----
        prim<P>(Us, a.gam_1, q);
        lds_put<NV>(Q, t, q);
        __syncthreads();
        lds_get<NV>(Q, tm, qm);
        lds_get<NV>(Q, tp, qp);
        faces<P, LIM>(a, qm, q, qp, fp, fm);
        lds_put<NV>(S, t, fm);
        __syncthreads();
        lds_get<NV>(S, tp, r);
        flux<P>(a, fp, r, F);
        lds_put<NV>(T, t, F);
        __syncthreads();
    }
    double dtb = 0.0, chb = 0.0;
    double fpb[NV];
    // ---- reverse: stage 2 ----
    {
        double lp[NV];  // lam' through the psi damping and the floors of stage 2
        {
            double U[NV], Fm[NV], R2[NV], Up[NV];
            load_u(U);
            lds_get<NV>(T, tm, Fm);
#pragma unroll
            for (int v = 0; v < NV; v++) {
                R2[v] = Fm[v] - F[v];
                const double un = U[v] + a.c2 * R2[v];
                Up[v] = (v < 5) ? un + 0.0 : un;
            }
#pragma unroll
            for (int k = 0; k < NV; k++) lp[k] = a.lam_out[(long long)plane_of_adj<DIR>(k) * a.sv + idx];
            if constexpr (P::MAG) lp[8] = lp[8] * a.psi_fac;
            floors_vjp<P>(a, Up, lp);
            if (outl) {
                double acc = 0.0;
#pragma unroll
                for (int v = 0; v < NV; v++) acc += lp[v] * R2[v];
                dtb += acc / a.dl;  // c2 = dt/dl
            }
        }
        lds_put<NV>(S, t, lp);
        __syncthreads();
        // interface k+1/2: fp is cell k's left state, r cell k+1's right state
        double lpn[NV], fb[NV], rb[NV];
        lds_get<NV>(S, tp, lpn);
#pragma unroll
        for (int v = 0; v < NV; v++) {
            fb[v] = a.c2 * (lpn[v] - lp[v]);
            fpb[v] = rb[v] = 0.0;
        }
        const double cb = flux_vjp<P>(a, fp, r, fb, fpb, rb);
        if (outl) chb += cb;
        lds_put<NV>(T, t, rb);  // belongs to cell k+1
    }
    __syncthreads();
    {
        double qb[NV], dlb[NV], drb[NV];
        {
            double fmb[NV], qc[NV], qm[NV], qp[NV];
            lds_get<NV>(T, tm, fmb);
            lds_get<NV>(Q, t, qc);
            lds_get<NV>(Q, tm, qm);
            lds_get<NV>(Q, tp, qp);
            faces_vjp<P, LIM>(a, qm, qc, qp, fpb, fmb, qb, dlb, drb);
        }
        __syncthreads();
        lds_put<NV>(T, t, dlb);
        lds_put<NV>(Q, t, drb);
        __syncthreads();
        lds_get<NV>(T, tp, dlb);
        lds_get<NV>(Q, tm, drb);
        double lsp[NV];  // lam* through the floors of stage 1
#pragma unroll
        for (int v = 0; v < NV; v++) {
            qb[v] += drb[v] - dlb[v];
            lsp[v] = 0.0;
        }
        double U[NV], R1[NV], W[NV];
        load_u(U);
        lds_get<NV>(K, t, R1);
        stage1(U, R1, W);
        floored(W);
        prim_vjp<P>(a, W, qb, lsp);
        stage1(U, R1, W);
        floors_vjp<P>(a, W, lsp);
        if (outl) {
            double acc = 0.0;
#pragma unroll
            for (int v = 0; v < NV; v++) acc += lsp[v] * R1[v];
            dtb += (0.5 * acc) / a.dl;  // c1 = (dt/2)/dl
        }
        lds_put<NV>(K, t, lsp);
        // S: the two direct terms lam' + lam* of the own cell
#pragma unroll
        for (int v = 0; v < NV; v++) S[t * NV + v] = lsp[v] + S[t * NV + v];
        double q[NV];
        prim<P>(U, a.gam_1, q);
        __syncthreads();
        lds_put<NV>(Q, t, q);
    }
    __syncthreads();
    // ---- reverse: stage 1 ----
    {
        double fb[NV], rb[NV];
        {
            double qm[NV], q[NV], qp[NV], fm[NV];
            lds_get<NV>(Q, tm, qm);
            lds_get<NV>(Q, t, q);
            lds_get<NV>(Q, tp, qp);
            faces<P, LIM>(a, qm, q, qp, fp, fm);
            lds_put<NV>(T, t, fm);
#pragma unroll
            for (int v = 0; v < NV; v++) {
                fb[v] = a.c1 * (K[tp * NV + v] - K[t * NV + v]);
                fpb[v] = rb[v] = 0.0;
            }
        }
        __syncthreads();
        lds_get<NV>(T, tp, r);
        const double cb = flux_vjp<P>(a, fp, r, fb, fpb, rb);
        if (outl) chb += cb;
        lds_put<NV>(K, t, rb);
    }
    __syncthreads();
    double lam[NV];
    {
        double qb[NV], dlb[NV], drb[NV], lsp[NV];
        {
            double fmb[NV], qc[NV], qm[NV], qp[NV];
            lds_get<NV>(K, tm, fmb);
            lds_get<NV>(Q, t, qc);
            lds_get<NV>(Q, tm, qm);
            lds_get<NV>(Q, tp, qp);
            faces_vjp<P, LIM>(a, qm, qc, qp, fpb, fmb, qb, dlb, drb);
        }
        lds_put<NV>(T, t, dlb);
        lds_get<NV>(S, t, lsp);
        lds_put<NV>(S, t, drb);
        __syncthreads();
        lds_get<NV>(T, tp, dlb);
        lds_get<NV>(S, tm, drb);
#pragma unroll
        for (int v = 0; v < NV; v++) {
            qb[v] += drb[v] - dlb[v];
            lam[v] = 0.0;
        }
        double U[NV];
        load_u(U);
        prim_vjp<P>(a, U, qb, lam);
#pragma unroll
        for (int v = 0; v < NV; v++) lam[v] = lam[v] + lsp[v];
    }
    if (outl) {
#pragma unroll
        for (int k = 0; k < NV; k++) a.lam_in[(long long)plane_of_adj<DIR>(k) * a.sv + idx] = lam[k];
    }
    // dL/d(dt) and dL/d(ch): per-wave sums in a fixed order, one slot per wave of the grid
    const int lane = t & 63;
    const int nact = min(64, nt - (t & ~63));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double o1 = __shfl_xor(dtb, o, 64);
        const double o2 = __shfl_xor(chb, o, 64);
        // the lower lane of each pair accumulates; lane 0 ends with the sum
        if ((lane ^ o) < nact && lane < (lane ^ o)) {
            dtb += o1;
            chb += o2;
        }
    }
    if (lane == 0) {
        const long long w = (long long)bid * ((nt + 63) / 64) + t / 64;
        a.dtb_part[w] = dtb;
        a.chb_part[w] = chb;
    }
}

template <int DIR, class P, int LIM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_sweep_adjoint(const AdjArgs a)
{
    extern __shared__ double lds[];
    // XCD-aware order, as k_sweep: tiles whose cells share cache lines (the
    // pencils of a y or z tile are a fraction of a line wide) share an L2
    adjoint_tile<DIR, P, LIM>(a, (int)xcd_order(), lds);
}

// Adjoint sweep over a block list (independent instances): as k_sweep_list, a
// tile per workgroup, per-block arguments from a table.
template <int DIR, class P, int LIM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_sweep_adjoint_list(const AdjListArgs L)
{
    extern __shared__ double lds[];
    typedef const __attribute__((address_space(4))) unsigned cu32;
    const unsigned item = L.item0 + xcd_order();
    const int blk = __builtin_amdgcn_readfirstlane((int)((cu32 *)L.items)[item]);
    AdjArgs a;
    static_assert(sizeof(AdjArgs) % 4 == 0, "AdjArgs is copied in dwords");
    cu32 *w = (cu32 *)(L.args + blk);
    unsigned *aw = reinterpret_cast<unsigned *>(&a);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(AdjArgs) / 4); i++) aw[i] = w[i];
    adjoint_tile<DIR, P, LIM>(a, (int)(item - ((cu32 *)L.first)[blk]), lds);
}

// Deterministic sum of n per-wave partials: kRedParts fixed ranges
// [n*g/kRedParts, n*(g+1)/kRedParts), each summed by one 256-lane workgroup
// (per-lane strided sums, then a tree), then the range sums added in order g.
// The kernels over many jobs use the same ranges and order, so both give the
// same bits.
__device__ double wg_range_sum(const double *__restrict__ part, long long lo, long long hi, double *red)
{
    const int t = threadIdx.x;
    double acc = 0.0;
    for (long long i = lo + t; i < hi; i += 256) acc += part[i];
    red[t] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) red[t] = red[t] + red[t + w];
        __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
}

__device__ __forceinline__ long long range_lo(long long n, int g) { return n * g / kRedParts; }

// range g of job j into part[n + g]: a workgroup per range.  (One workgroup
// per job walked its 64 ranges one after the other, ten barriers each: 61 us
// for the 40 sums of 20 instances.)
__device__ __forceinline__ void sum_range(const SumJob &j, int g)
{
    __shared__ double red[256];
    const double r = wg_range_sum(j.part, range_lo(j.n, g), range_lo(j.n, g + 1), red);
    if (threadIdx.x == 0) j.part[j.n + g] = r;
}

// the range sums of job j in order: a wave fetches them, one lane adds
__device__ __forceinline__ void sum_final(const SumJob &j)
{
    static_assert(kRedParts == 64, "a range sum per lane");
    __shared__ double v[kRedParts];
    v[threadIdx.x] = j.part[j.n + threadIdx.x];
    __syncthreads();
    if (threadIdx.x != 0) return;
    double tot = 0.0;
#pragma unroll
    for (int g = 0; g < kRedParts; g++) tot += v[g];
    j.out[0] = tot;
}

// The sums of all sweeps of a step (and of all instances) in two launches.
// After every sweep they were two launches of 5 us each, which nothing
// overlaps: 172 of the 1590 us of a 3-step gradient of a 45x40x34 MHD block.
__global__ __launch_bounds__(256) void k_sum_ranges_jobs(const SumJob *__restrict__ jobs)
{
    sum_range(jobs[blockIdx.y], blockIdx.x);
}
__global__ __launch_bounds__(64) void k_sum_final_jobs(const SumJob *__restrict__ jobs) { sum_final(jobs[blockIdx.x]); }
__global__ __launch_bounds__(256) void k_sum_ranges(const SweepSums s) { sum_range(s.job[blockIdx.y], blockIdx.x); }
__global__ __launch_bounds__(64) void k_sum_final(const SweepSums s) { sum_final(s.job[blockIdx.x]); }

__global__ void k_zero_best(unsigned long long *best)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *best = ~0ull;
}

// timestep adjoint: the cell and direction where dl_d/c_d is smallest (the
// smallest linear index among exact ties), then dL/dU there.
__device__ __forceinline__ double cell_cs(const DtAdjArgs &a, const double *u)
{
    const double d = u[0], e = u[4 * a.sv];
    const double m0 = u[a.sv], m1 = u[2 * a.sv], m2 = u[3 * a.sv];
    const double ek = (0.5 * ((m0 * m0 + m1 * m1) + m2 * m2)) / d;
    if (a.magnetized) {
        const double bx = u[5 * a.sv], by = u[6 * a.sv], bz = u[7 * a.sv];
        const double pmag = 0.5 * ((bx * bx + by * by) + bz * bz);
        const double ps = (e - ek) * a.gam_1 + (2.0 - a.gam) * pmag;
        const double pr = ps - pmag;
        return sqrt(fabs((2.0 * pmag + a.gam * pr) / d));
    }
    const double pr = (e - ek) * a.gam_1;
    return sqrt(fabs((a.gam * pr) / d));
}

__global__ __launch_bounds__(256) void k_dt_argmin(const DtAdjArgs a, unsigned long long *best)
{
    const long long ncell = (long long)a.n[0] * a.n[1] * a.n[2];
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell;
         c += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(c % a.n[0]);
        const long long r = c / a.n[0];
        const int j = (int)(r % a.n[1]);
        const int k = (int)(r / a.n[1]);
        const long long idx =
            (long long)(i + a.g[0]) + (long long)a.sy * (j + a.g[1]) + (long long)a.sz * (k + a.g[2]);
        const double *u = a.u + idx;
        const double d = u[0];
        const double cs = cell_cs(a, u);
        for (int q = 0; q < 3; q++) {
            if (!a.has_dir[q]) continue;
            const double v = (d > 0.0) ? fabs(u[(1 + q) * a.sv] / d) : 0.0;
            const double cc = fmx(v + cs, 1.17549435082228750797e-38);
            if (a.dl[q] / cc == a.mn) atomicMin(best, (unsigned long long)(c * 3 + q));
        }
    }
}

__device__ void k_dt_apply_body(const DtAdjArgs &a, const unsigned long long *best, double *lam)
{
    const unsigned long long b = *best;
    if (b == ~0ull) return;
    const long long c = (long long)(b / 3);
    const int q = (int)(b % 3);
    const int i = (int)(c % a.n[0]);
    const long long r = c / a.n[0];
    const int j = (int)(r % a.n[1]);
    const int k = (int)(r / a.n[1]);
    const long long idx = (long long)(i + a.g[0]) + (long long)a.sy * (j + a.g[1]) + (long long)a.sz * (k + a.g[2]);
    // dt = cfl * dl_q / c_q
    if (a.magnetized) {
        double u[9], ub[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        for (int v = 0; v < 9; v++) u[v] = a.u[(long long)v * a.sv + idx];
        dt_vjp_mhd(u, q, a.dl[q], a.gam, a.gam_1, a.cfl * a.dtb, ub);
        for (int v = 0; v < 8; v++) lam[(long long)v * a.sv + idx] += ub[v];
    } else {
        double u[5], ub[5] = {0, 0, 0, 0, 0};
        for (int v = 0; v < 5; v++) u[v] = a.u[(long long)v * a.sv + idx];
        dt_vjp_hd(u, q, a.dl[q], a.gam, a.gam_1, a.cfl * a.dtb, ub);
        for (int v = 0; v < 5; v++) lam[(long long)v * a.sv + idx] += ub[v];
    }
}

__global__ void k_dt_apply(const DtAdjArgs a, const unsigned long long *best, double *lam)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    k_dt_apply_body(a, best, lam);
}

__global__ void k_dt_init_jobs(const DtBatchJob *__restrict__ jobs, int njobs)
{
    const int jb = blockIdx.x * blockDim.x + threadIdx.x;
    if (jb >= njobs) return;
    *jobs[jb].mn = 1.7976931348623157e308;
    *jobs[jb].best = ~0ull;
}

// grid (chunks, jobs): min over the job's cells and directions of dl/c
// (positive: ordered as its bit pattern).  (A workgroup per job took 320 us
// for the largest of 20 instances, 256^2 cells.)
__global__ __launch_bounds__(256) void k_dt_mn_jobs(const DtBatchJob *__restrict__ jobs)
{
    const DtBatchJob &J = jobs[blockIdx.y];
    const DtAdjArgs &a = J.a;
    const long long ncell = (long long)a.n[0] * a.n[1] * a.n[2];
    if ((long long)blockIdx.x * 256 >= ncell) return;
    double m = 1.7976931348623157e308;
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell;
         c += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(c % a.n[0]);
        const long long r = c / a.n[0];
        const int j = (int)(r % a.n[1]);
        const int k = (int)(r / a.n[1]);
        const long long idx =
            (long long)(i + a.g[0]) + (long long)a.sy * (j + a.g[1]) + (long long)a.sz * (k + a.g[2]);
        const double *u = a.u + idx;
        const double d = u[0];
        const double cs = cell_cs(a, u);
        for (int q = 0; q < 3; q++) {
            if (!a.has_dir[q]) continue;
            const double v = (d > 0.0) ? fabs(u[(1 + q) * a.sv] / d) : 0.0;
            m = fmn(m, a.dl[q] / fmx(v + cs, 1.17549435082228750797e-38));
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmn(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0)
        atomicMin((unsigned long long *)J.mn, (unsigned long long)__double_as_longlong(m));
}

// grid (chunks, jobs): the smallest cell/direction index attaining the minimum
__global__ __launch_bounds__(256) void k_dt_argmin_jobs(const DtBatchJob *__restrict__ jobs)
{
    const DtBatchJob &J = jobs[blockIdx.y];
    const DtAdjArgs &a = J.a;
    const double mn = *J.mn;
    const long long ncell = (long long)a.n[0] * a.n[1] * a.n[2];
    for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell;
         c += (long long)gridDim.x * blockDim.x) {
        const int i = (int)(c % a.n[0]);
        const long long r = c / a.n[0];
        const int j = (int)(r % a.n[1]);
        const int k = (int)(r / a.n[1]);
        const long long idx =
            (long long)(i + a.g[0]) + (long long)a.sy * (j + a.g[1]) + (long long)a.sz * (k + a.g[2]);
        const double *u = a.u + idx;
        const double d = u[0];
        const double cs = cell_cs(a, u);
        for (int q = 0; q < 3; q++) {
            if (!a.has_dir[q]) continue;
            const double v = (d > 0.0) ? fabs(u[(1 + q) * a.sv] / d) : 0.0;
            if (a.dl[q] / fmx(v + cs, 1.17549435082228750797e-38) == mn)
                atomicMin(J.best, (unsigned long long)(c * 3 + q));
        }
    }
}

// one thread per job
__global__ void k_dt_apply_jobs(const DtBatchJob *__restrict__ jobs, int njobs)
{
    const int jb = blockIdx.x * blockDim.x + threadIdx.x;
    if (jb >= njobs) return;
    const DtBatchJob &J = jobs[jb];
    DtAdjArgs a = J.a;
    a.dtb = J.dtb;
    k_dt_apply_body(a, J.best, J.lam);
}

// ---- launchers ------------------------------------------------------------------

template <int DIR, class P, int LIM>
static hipError_t adj_t(const AdjArgs &a, int nt, long long nblk, hipStream_t st)
{
    const size_t lds = sizeof(double) * kAdjArrays * P::NV * nt;
    static bool raised = false;
    if (!raised) {
        hipError_t e = hipFuncSetAttribute((const void *)k_sweep_adjoint<DIR, P, LIM>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        raised = true;
    }
    if (lds > 160 * 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_sweep_adjoint<DIR, P, LIM>), dim3((unsigned)nblk), dim3(nt), lds, st, a);
    return hipGetLastError();
}

template <int DIR, class P>
static hipError_t adj_lim(const AdjArgs &a, int nt, long long nblk, hipStream_t st)
{
    if (a.lim == a.limb || !P::MAG) {
        switch (a.lim) {
        case LIM_VANLEER: return adj_t<DIR, P, LIM_VANLEER>(a, nt, nblk, st);
        case LIM_MINMOD: return adj_t<DIR, P, LIM_MINMOD>(a, nt, nblk, st);
        case LIM_MONCEN: return adj_t<DIR, P, LIM_MONCEN>(a, nt, nblk, st);
        case LIM_SUPERBEE: return adj_t<DIR, P, LIM_SUPERBEE>(a, nt, nblk, st);
        default: return hipErrorInvalidValue;
        }
    }
    return adj_t<DIR, P, -1>(a, nt, nblk, st);
}

template <int DIR, class P, int LIM>
static hipError_t adjl_t(const AdjListArgs &L, hipStream_t st)
{
    const int nt = 256;
    const void *fn = (const void *)k_sweep_adjoint_list<DIR, P, LIM>;
    const size_t lds = sizeof(double) * kAdjArrays * P::NV * nt;
    const size_t lds_max = 160 * 1024;
    static bool raised = false;
    if (!raised) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_max);
        if (e != hipSuccess) return e;
        raised = true;
    }
    if (lds > lds_max) return hipErrorInvalidValue;
    AdjListArgs l = L;
    for (l.item0 = 0; l.item0 < L.nitems; l.item0 += kListPiece) {
        const unsigned n = L.nitems - l.item0 < kListPiece ? L.nitems - l.item0 : kListPiece;
        hipLaunchKernelGGL((k_sweep_adjoint_list<DIR, P, LIM>), dim3(n), dim3(nt), lds, st, l);
        if (l.item0 + n == L.nitems) break;  // (the next item0 may not fit 32 bits)
    }
    return hipGetLastError();
}

template <int DIR, class P>
static hipError_t adjl_lim(int lim, int limb, const AdjListArgs &L, hipStream_t st)
{
    if (lim == limb || !P::MAG) {
        switch (lim) {
        case LIM_VANLEER: return adjl_t<DIR, P, LIM_VANLEER>(L, st);
        case LIM_MINMOD: return adjl_t<DIR, P, LIM_MINMOD>(L, st);
        case LIM_MONCEN: return adjl_t<DIR, P, LIM_MONCEN>(L, st);
        case LIM_SUPERBEE: return adjl_t<DIR, P, LIM_SUPERBEE>(L, st);
        default: return hipErrorInvalidValue;
        }
    }
    return adjl_t<DIR, P, -1>(L, st);
}

static hipError_t adjl_dispatch(int dir, bool mhd, int lim, int limb, const AdjListArgs &L, hipStream_t st)
{
    if (mhd) {
        if (dir == 0) return adjl_lim<0, MHD>(lim, limb, L, st);
        if (dir == 1) return adjl_lim<1, MHD>(lim, limb, L, st);
        if (dir == 2) return adjl_lim<2, MHD>(lim, limb, L, st);
    } else {
        if (dir == 0) return adjl_lim<0, HD>(lim, limb, L, st);
        if (dir == 1) return adjl_lim<1, HD>(lim, limb, L, st);
        if (dir == 2) return adjl_lim<2, HD>(lim, limb, L, st);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_sweep_adjoint_list(int dir, bool mhd, int lim, int limb, const AdjListArgs &L, hipStream_t st)
{
    return adjl_dispatch(dir, mhd, lim, limb, L, st);
}

hipError_t launch_sum_parts_jobs(const SumJob *jobs, int njobs, hipStream_t st)
{
    if (njobs <= 0) return hipSuccess;
    for (int j0 = 0; j0 < njobs; j0 += 32768) {
        const int n = njobs - j0 < 32768 ? njobs - j0 : 32768;
        hipLaunchKernelGGL(k_sum_ranges_jobs, dim3(kRedParts, (unsigned)n), dim3(256), 0, st, jobs + j0);
    }
    hipLaunchKernelGGL(k_sum_final_jobs, dim3((unsigned)njobs), dim3(64), 0, st, jobs);
    return hipGetLastError();
}

hipError_t launch_sweep_sums(const SweepSums &s, int njobs, hipStream_t st)
{
    if (njobs < 1 || njobs > 2 * kStepSweeps) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sum_ranges, dim3(kRedParts, (unsigned)njobs), dim3(256), 0, st, s);
    hipLaunchKernelGGL(k_sum_final, dim3((unsigned)njobs), dim3(64), 0, st, s);
    return hipGetLastError();
}

template <class P>
static hipError_t adj_dir(int dir, const AdjArgs &a, int nt, long long nblk, hipStream_t st)
{
    if (dir == 0) return adj_lim<0, P>(a, nt, nblk, st);
    if (dir == 1) return adj_lim<1, P>(a, nt, nblk, st);
    if (dir == 2) return adj_lim<2, P>(a, nt, nblk, st);
    return hipErrorInvalidValue;
}

// Every adjoint tile runs on a 256-lane workgroup (lanes past TP*TS idle),
// as in the list kernel: four partial slots per tile in both, so
// their sums of the same partials agree bit for bit.
long long sweep_adjoint_parts(const AdjArgs &a) { return (long long)a.chunks * a.ptiles * 4; }

hipError_t launch_sweep_adjoint(int dir, bool mhd, const AdjArgs &a, hipStream_t st)
{
    const int nt = 256;
    if (a.TP * a.TS < 1 || a.TP * a.TS > nt || a.out < 1 || a.out != a.TS - 16) return hipErrorInvalidValue;
    const long long nblk = (long long)a.chunks * a.ptiles;
    return mhd ? adj_dir<MHD>(dir, a, nt, nblk, st) : adj_dir<HD>(dir, a, nt, nblk, st);
}

hipError_t launch_dt_adjoint_batch(const DtBatchJob *jobs, int njobs, hipStream_t st)
{
    if (njobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dt_init_jobs, dim3((unsigned)((njobs + 63) / 64)), dim3(64), 0, st, jobs, njobs);
    for (int j0 = 0; j0 < njobs; j0 += 32768) {
        const unsigned n = (unsigned)(njobs - j0 < 32768 ? njobs - j0 : 32768);
        hipLaunchKernelGGL(k_dt_mn_jobs, dim3(64, n), dim3(256), 0, st, jobs + j0);
        hipLaunchKernelGGL(k_dt_argmin_jobs, dim3(64, n), dim3(256), 0, st, jobs + j0);
    }
    hipLaunchKernelGGL(k_dt_apply_jobs, dim3((unsigned)((njobs + 63) / 64)), dim3(64), 0, st, jobs, njobs);
    return hipGetLastError();
}

hipError_t launch_dt_adjoint(const DtAdjArgs &a, unsigned long long *best, double *lam, hipStream_t st)
{
    hipLaunchKernelGGL(k_zero_best, dim3(1), dim3(1), 0, st, best);
    const long long ncell = (long long)a.n[0] * a.n[1] * a.n[2];
    long long blocks = (ncell + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(k_dt_argmin, dim3((unsigned)blocks), dim3(256), 0, st, a, best);
    hipLaunchKernelGGL(k_dt_apply, dim3(1), dim3(64), 0, st, a, best, lam);
    return hipGetLastError();
}

}  // namespace pk
