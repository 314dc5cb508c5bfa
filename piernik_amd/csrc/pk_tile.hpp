// pk_tile.hpp -- device pieces of the split and unsplit tiles: variable order,
// LDS layout, index arithmetic and the timestep of the cells written.
// Included inside namespace PK_KNS, after pk_math.hpp: both builds (exact and
// relaxed arithmetic) get their own copy.
#pragma once

template <int DIR>
__device__ __forceinline__ int plane_of(int k)
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

// One lane's NV values in an LDS array of the tile, lane by lane (NV is odd,
// so consecutive lanes fall on different banks): one address per lane and
// neighbour, the variables at immediate offsets, read two at a time.
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

// Cell index c along the sweep (ghosts included) -> the interior cell a ghost
// of a block periodic on itself copies (wrap: the sweep reads those instead of
// the ghosts, which it leaves as they are).
__device__ __forceinline__ int wrap_cell(int c, int g, int n)
{
    return c < g ? c + n : (c >= g + n ? c - n : c);
}

// q = t / d for 0 <= t < 512 and 1 <= d <= 512: (t + 1/2) / d is at least
// 1/(2 d) > 9e-4 away from a whole number, far more than the roundings of the
// reciprocal and the product (below 2e-4 at 512); an integer division takes
// three times the instructions.
__device__ __forceinline__ int small_div(int t, int d)
{
    return (int)(((float)t + 0.5f) * __builtin_amdgcn_rcpf((float)d));
}

// timestep_fluid (timestep.F90:460-490, ion_cs / neu_cs) of one written
// cell, folded into a lane's running min of dl/c per direction and max of c.
template <int DIR, class P, class ARGS>
__device__ __forceinline__ void dt_cell(const ARGS &a, const double (&Wn)[P::NV], double (&mn)[3], double &cmax)
{
    const double small = 1.17549435082228750797e-38;
    const double d = Wn[0];
    const double mx = Wn[plane_of<DIR>(1)], my = Wn[plane_of<DIR>(2)], mz = Wn[plane_of<DIR>(3)];
    const double e = Wn[4];
    const double m[3] = {mx, my, mz};
    double v[3] = {0.0, 0.0, 0.0};
    if (d > 0.0) {
#pragma unroll
        for (int q = 0; q < 3; q++) v[q] = fabs(qdiv(m[q], d));
    }
    const double ek = qdiv(0.5 * ((mx * mx + my * my) + mz * mz), d);
    double cs;
    if constexpr (P::MAG) {
        const double bx = Wn[plane_of<DIR>(5)], by = Wn[plane_of<DIR>(6)], bz = Wn[plane_of<DIR>(7)];
        const double pmag = 0.5 * ((bx * bx + by * by) + bz * bz);
        const double ps = (e - ek) * a.gam_1 + (2.0 - a.gam) * pmag;
        const double pr = ps - pmag;
        cs = qsqrt(fabs(qdiv(2.0 * pmag + a.gam * pr, d)));
    } else {
        const double pr = (e - ek) * a.gam_1;
        cs = qsqrt(fabs(qdiv(a.gam * pr, d)));
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double c = fmx(v[q] + cs, small);
        cmax = fmx(cmax, c);
        if (a.has_dir[q]) mn[q] = fmn(mn[q], qdiv(a.dl[q], c));
    }
}

// The lanes' running values reduced over the wave and folded into one slot
// with 64-bit atomics (the values are positive, so their bit patterns order
// as the numbers do; min and max do not depend on the order of reduction).
template <class ARGS>
__device__ __forceinline__ void dt_reduce(const ARGS &a, double (&mn)[3], double &cmax, unsigned slot_id)
{
    // xor butterfly over the lanes that exist (the last wave of a workgroup
    // may be partial); partners beyond it are skipped, lane 0 ends with all.
    const int lane = threadIdx.x & 63;
    const int nact = min(64, (int)blockDim.x - (int)(threadIdx.x & ~63u));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const bool take = (lane ^ o) < nact;
        double t[4];
#pragma unroll
        for (int q = 0; q < 3; q++) t[q] = __shfl_xor(mn[q], o, 64);
        t[3] = __shfl_xor(cmax, o, 64);
        if (take) {
#pragma unroll
            for (int q = 0; q < 3; q++) mn[q] = fmn(mn[q], t[q]);
            cmax = fmx(cmax, t[3]);
        }
    }
    if ((threadIdx.x & 63) == 0) {
        const int slot = (int)((slot_id * (blockDim.x / 64u) + threadIdx.x / 64u) % (unsigned)a.nslots);
        unsigned long long *s = a.dtslots + 4 * slot;
#pragma unroll
        for (int q = 0; q < 3; q++) atomicMin(s + q, (unsigned long long)__double_as_longlong(mn[q]));
        atomicMax(s + 3, (unsigned long long)__double_as_longlong(cmax));
    }
}
