// pk_blocks.hip -- gfx950 kernels over whole blocks and block lists: layout
// conversion at the boundary, ghost refresh and exchange, the standalone
// timestep reduction and the bookkeeping of the list launches.  Compiled
// without FMA contraction (the timestep formula rounds as the reference's).
#include <hip/hip_runtime.h>
#include "pk_math.hpp"
#include "pk_kernels.hpp"

namespace pk {

__global__ void k_fill_items(const unsigned *__restrict__ first, int nblocks, unsigned *__restrict__ items)
{
    // one workgroup per block writes its range of the item table
    const int b = blockIdx.x;
    if (b >= nblocks) return;
    for (unsigned i = first[b] + threadIdx.x; i < first[b + 1]; i += blockDim.x) items[i] = (unsigned)b;
}

// a batch of device-to-device copies: workgroups stride over the jobs
__global__ __launch_bounds__(256) void k_copy_blocks(const CopyJob *__restrict__ jobs, int njobs)
{
    for (int j = blockIdx.y; j < njobs; j += gridDim.y) {
        const CopyJob c = jobs[j];
        for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < c.n;
             i += (long long)gridDim.x * blockDim.x)
            c.dst[i] = c.src[i];
    }
}

__global__ void k_zero_u32(unsigned *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

__global__ void k_scale(double *__restrict__ x, long long n, double fac)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] * fac;
}

// timestep_fluid (timestep.F90:460-490) with ion_cs / neu_cs
// (initionized.F90:137-141, initneutral.F90:102-105) of cell c of the
// block's interior (x fastest), folded into the running min of dl_d/c_d for
// d = x, y, z and max of c.
template <bool MAG>
__device__ __forceinline__ void dt_fold(const DtArgs &a, unsigned c, double (&m)[3], double &cmax)
{
    const unsigned nx = (unsigned)a.n[0], ny = (unsigned)a.n[1];
    const unsigned r = c / nx, i = c - r * nx;
    const unsigned k = r / ny, j = r - k * ny;
    const long long idx = (long long)(i + a.g[0]) + (long long)a.sy * (j + a.g[1]) + (long long)a.sz * (k + a.g[2]);
    const double *u = a.u + (long long)a.plane0 * a.sv + idx;
    const double d = u[0], mx = u[a.sv], my = u[2 * a.sv], mz = u[3 * a.sv], e = u[4 * a.sv];
    double v[3] = {0.0, 0.0, 0.0};
    if (d > 0.0) {
        v[0] = fabs(qdiv(mx, d));
        v[1] = fabs(qdiv(my, d));
        v[2] = fabs(qdiv(mz, d));
    }
    const double ek = qdiv(0.5 * ((mx * mx + my * my) + mz * mz), d);
    double cs;
    if (MAG) {
        const double *b = a.u + (long long)a.bplane * a.sv + idx;
        const double bx = b[0], by = b[a.sv], bz = b[2 * a.sv];
        const double pmag = 0.5 * ((bx * bx + by * by) + bz * bz);
        const double ps = (e - ek) * a.gam_1 + (2.0 - a.gam) * pmag;
        const double pr = ps - pmag;
        cs = qsqrt(fabs(qdiv(2.0 * pmag + a.gam * pr, d)));
    } else {
        const double pr = (e - ek) * a.gam_1;
        cs = qsqrt(fabs(qdiv(a.gam * pr, d)));
    }
    const double small = 1.17549435082228750797e-38;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double cq = fmx(v[q] + cs, small);
        cmax = fmx(cmax, cq);
        if (a.has_dir[q]) m[q] = fmn(m[q], qdiv(a.dl[q], cq));
    }
}

// min and max over the lanes of a whole wave
__device__ __forceinline__ void wave_minmax(double (&m)[3], double &cmax)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
#pragma unroll
        for (int q = 0; q < 3; q++) m[q] = fmn(m[q], __shfl_xor(m[q], o, 64));
        cmax = fmx(cmax, __shfl_xor(cmax, o, 64));
    }
}

// Results of a 256-lane workgroup's four waves in lane 0 of its first one.
__device__ __forceinline__ void wg_minmax(double (&m)[3], double &cmax)
{
    __shared__ double red[4][4];
    wave_minmax(m, cmax);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        for (int q = 0; q < 3; q++) red[q][w] = m[q];
        red[3][w] = cmax;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; k++) {
            for (int q = 0; q < 3; q++) m[q] = fmn(m[q], red[q][k]);
            cmax = fmx(cmax, red[3][k]);
        }
    }
}

// Per-workgroup partial results of one block of fewer than 2^32 cells (a
// state of 2^32 cells would take 160 GiB per buffer; launch_dt checks).
template <bool MAG>
__global__ __launch_bounds__(256) void k_dt_partial(const DtArgs a, double *__restrict__ part)
{
    const double huge = 1.7976931348623157e308;
    double m[3] = {huge, huge, huge}, cmax = 1.17549435082228750797e-38;
    const unsigned ncell = (unsigned)a.n[0] * (unsigned)a.n[1] * (unsigned)a.n[2];
    for (unsigned long long c = (unsigned long long)blockIdx.x * 256u + threadIdx.x; c < ncell; c += (unsigned long long)gridDim.x * 256u)
        dt_fold<MAG>(a, (unsigned)c, m, cmax);
    wg_minmax(m, cmax);
    if (threadIdx.x == 0) {
        part[4 * blockIdx.x + 0] = m[0];
        part[4 * blockIdx.x + 1] = m[1];
        part[4 * blockIdx.x + 2] = m[2];
        part[4 * blockIdx.x + 3] = cmax;
    }
}

__global__ __launch_bounds__(256) void k_dt_final(const double *__restrict__ part, int nparts,
                                                  double *__restrict__ out)
{
    const double huge = 1.7976931348623157e308;
    double m[3] = {huge, huge, huge}, cmax = 0.0;
    for (int i = threadIdx.x; i < nparts; i += 256) {
        for (int q = 0; q < 3; q++) m[q] = fmn(m[q], part[4 * i + q]);
        cmax = fmx(cmax, part[4 * i + 3]);
    }
    wg_minmax(m, cmax);
    if (threadIdx.x == 0) {
        out[0] = m[0];
        out[1] = m[1];
        out[2] = m[2];
        out[3] = cmax;
    }
}

// timestep_fluid of every block and fluid of a list in one launch: grid
// (chunks, jobs), job j's results folded into the slots of its block
// (per_block) or of the whole list; min and max do not depend on the order,
// and positive doubles order as their bit patterns.  One launch in place of
// two and a host wait per block: the first step of 144 two-fluid blocks spent
// 288 launches and 144 waits on it.
__global__ __launch_bounds__(256) void k_dt_list(const DtArgs *__restrict__ jobs, int nfl, unsigned long long *slots,
                                                 int nslots, int per_block)
{
    const DtArgs &a = jobs[blockIdx.y];
    const double huge = 1.7976931348623157e308;
    double m[3] = {huge, huge, huge}, cmax = 1.17549435082228750797e-38;
    const unsigned ncell = (unsigned)a.n[0] * (unsigned)a.n[1] * (unsigned)a.n[2];
    if ((unsigned long long)blockIdx.x * 256u >= ncell) return;
    for (unsigned long long c = (unsigned long long)blockIdx.x * 256u + threadIdx.x; c < ncell; c += (unsigned long long)gridDim.x * 256u) {
        if (a.magnetized)
            dt_fold<true>(a, (unsigned)c, m, cmax);
        else
            dt_fold<false>(a, (unsigned)c, m, cmax);
    }
    wg_minmax(m, cmax);
    if (threadIdx.x != 0) return;
    const unsigned blk = blockIdx.y / nfl;
    unsigned long long *s = slots + (per_block ? 4ull * nslots * blk : 0ull) +
                            4ull * ((blockIdx.x + (per_block ? 0u : 7u * blockIdx.y)) % (unsigned)nslots);
    for (int q = 0; q < 3; q++) atomicMin(s + q, (unsigned long long)__double_as_longlong(m[q]));
    atomicMax(s + 3, (unsigned long long)__double_as_longlong(cmax));
}

// ---- timestep slots ------------------------------------------------------------
// A sweep folds timestep_fluid of the cells it writes into slots of four
// 64-bit patterns; the final kernel reduces them and leaves them clean for
// the next reduction (no separate initialisation per step).

__device__ __forceinline__ void slot_clear(unsigned long long *s)
{
    const unsigned long long huge = (unsigned long long)__double_as_longlong(1.7976931348623157e308);
    s[0] = huge;
    s[1] = huge;
    s[2] = huge;
    s[3] = 0ull;
}

__global__ void k_dtslots_init(unsigned long long *slots, int nslots)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nslots) slot_clear(slots + 4ll * i);
}

// one workgroup per set of nslots slots: its four results, into device or
// pinned host memory
__global__ __launch_bounds__(256) void k_dtslots_final(unsigned long long *__restrict__ slots, int nslots,
                                                       double *__restrict__ out)
{
    unsigned long long *s = slots + 4ll * nslots * blockIdx.x;
    const double huge = 1.7976931348623157e308;
    double m[3] = {huge, huge, huge}, cmax = 0.0;
    for (int i = threadIdx.x; i < nslots; i += 256) {
        for (int q = 0; q < 3; q++) m[q] = fmn(m[q], __longlong_as_double((long long)s[4 * i + q]));
        cmax = fmx(cmax, __longlong_as_double((long long)s[4 * i + 3]));
        slot_clear(s + 4 * i);
    }
    wg_minmax(m, cmax);
    if (threadIdx.x == 0) {
        double *o = out + 4 * blockIdx.x;
        o[0] = m[0];
        o[1] = m[1];
        o[2] = m[2];
        o[3] = cmax;
    }
}

// ---- ghosts ------------------------------------------------------------------------

// The planes of one cell in as few groups of loads as they fit (a block has 5
// or 9 planes with one fluid, 10 or 14 with two).
__device__ __forceinline__ void copy_cell(const double *s, long long ssv, double *d, long long dsv, int np)
{
    if (np == 9)
        copy_planes<9>(s, ssv, d, dsv, np);
    else if (np == 14)
        copy_planes<14>(s, ssv, d, dsv, np);
    else
        copy_planes<5>(s, ssv, d, dsv, np);
}

// Ghost exchange between blocks (internal_boundaries_local,
// cg_list_bnd.F90:269-322): one job per face, cut into chunks of kFaceCells
// cells, one workgroup per chunk (wgjob names its job); cells run x fastest,
// so rows of y and z faces are coalesced, and a lane finds its cell once for
// all planes.  The time is latency, so a lane has one cell and its planes'
// loads are in flight together: an exchange of twelve 40x48x40 MHD blocks took
// 20 us a value at a time (1484 instructions per wave, 90 % of them index
// divisions), 17 with two cells a lane in groups of five planes, 14.6 so.
__global__ __launch_bounds__(256) void k_exchange_faces(const FaceJob *__restrict__ jobs, const int *__restrict__ wgjob)
{
    const FaceJob &J = jobs[wgjob[blockIdx.x]];
    const int e0 = J.ext[0], e01 = e0 * J.ext[1], ncell = e01 * J.ext[2];
    const int c = ((int)blockIdx.x - J.wg0) * kFaceCells + (int)threadIdx.x;
    if (c >= ncell) return;
    const int k = c / e01, r = c - k * e01;
    const int j = r / e0, i = r - j * e0;
    const double *s = J.src + (J.sorg[0] + i) + (long long)J.ssy * (J.sorg[1] + j) + (long long)J.ssz * (J.sorg[2] + k);
    double *d = J.dst + (J.dorg[0] + i) + (long long)J.dsy * (J.dorg[1] + j) + (long long)J.dsz * (J.dorg[2] + k);
    copy_cell(s, J.ssv, d, J.dsv, J.nplanes);
}
static_assert(kFaceCells == 256, "k_exchange_faces: a cell per lane");

// Periodic refresh of every ghost cell of a block in one launch: each ghost
// is a copy of the interior cell its coordinates wrap to, which is what
// refreshes along x, y and z in turn leave (n >= g).
__global__ __launch_bounds__(256) void k_fill_periodic(const GhostArgs a)
{
    const unsigned n[3] = {(unsigned)a.n[0], (unsigned)a.n[1], (unsigned)a.n[2]};
    const unsigned g[3] = {(unsigned)a.g[0], (unsigned)a.g[1], (unsigned)a.g[2]};
    unsigned c[3], f[3];
    if (!ghost_cell(blockIdx.x * 256u + threadIdx.x, n, g, c)) return;
#pragma unroll
    for (int d = 0; d < 3; d++) f[d] = c[d] < g[d] ? c[d] + n[d] : (c[d] >= g[d] + n[d] ? c[d] - n[d] : c[d]);
    double *base = a.u + (long long)a.plane0 * a.sv;
    copy_cell(base + f[0] + (long long)a.sy * f[1] + (long long)a.sz * f[2], a.sv,
              base + c[0] + (long long)a.sy * c[1] + (long long)a.sz * c[2], a.sv, a.nplanes);
}

// ---- layout conversion ---------------------------------------------------------------
// Arrays of the reference layout (variable fastest; up to three of them, for
// u, B and psi) <-> device planes, a cell per lane and every array in one
// launch: grid (cells of a z plane / 256, nz).  Bound by memory: 5.6 TB/s of
// 16 B per value at 256^3 (the strided accesses of a wave share cache lines).
// On small blocks the time is the latency of one lane's accesses, so the
// values of a cell are read in groups of up to kPl before they are written:
// one after another, 14 values of a cell of two fluids took 22 us to the planes'
// arrays and 14 us back on blocks of 85000 cells (a launch is 3 us).

// One array of a cell.
constexpr int kPl = 5;
template <bool IN>
__device__ __forceinline__ void planes_array(const PlaneMap &m, double *q, double *s, long long sv)
{
    for (int c0 = 0; c0 < m.nc; c0 += kPl) {
        double x[kPl];
#pragma unroll
        for (int c = 0; c < kPl; c++) {
            const int cc = min(c0 + c, m.nc - 1);
            x[c] = IN ? q[cc] : s[(long long)m.planes[cc] * sv];
        }
#pragma unroll
        for (int c = 0; c < kPl; c++) {
            if (c0 + c >= m.nc) break;
            (IN ? s[(long long)m.planes[c0 + c] * sv] : q[c0 + c]) = x[c];
        }
    }
}

template <bool IN>
__global__ __launch_bounds__(256) void k_planes(const PlanesArgs a)
{
    const unsigned nx = (unsigned)a.nx, ny = (unsigned)a.ny, nz = (unsigned)a.nz;
    const unsigned e = blockIdx.x * 256u + threadIdx.x;
    if (e >= nx * ny) return;
    const unsigned y = e / nx, x = e - y * nx;
    for (unsigned z = blockIdx.y; z < nz; z += gridDim.y) {
        const long long i = (long long)e + (long long)z * nx * ny;
        double *s = a.soa + x + (long long)a.sy * y + (long long)a.sz * z;
        // u of one fluid with B and psi: all nine values in flight
        if (a.aos[0] && a.aos[1] && a.aos[2] && a.map[0].nc == 5 && a.map[1].nc == 3 && a.map[2].nc == 1) {
            double *q[9], *p[9], v[9];
#pragma unroll
            for (int c = 0; c < 9; c++) {
                const int k = c < 5 ? 0 : (c < 8 ? 1 : 2), cc = c < 5 ? c : (c < 8 ? c - 5 : 0);
                q[c] = a.aos[k] + i * (k == 0 ? 5 : (k == 1 ? 3 : 1)) + cc;
                p[c] = s + (long long)a.map[k].planes[cc] * a.sv;
            }
#pragma unroll
            for (int c = 0; c < 9; c++) v[c] = IN ? *q[c] : *p[c];
#pragma unroll
            for (int c = 0; c < 9; c++) (IN ? *p[c] : *q[c]) = v[c];
            continue;
        }
#pragma unroll
        for (int k = 0; k < 3; k++)
            if (a.aos[k]) planes_array<IN>(a.map[k], a.aos[k] + i * a.map[k].nc, s, a.sv);
    }
}

// The adjoint of the periodic ghost refresh while converting: an interior
// cell's adjoint is its own plus those of the ghosts that copy it (folded
// along z, then y, then x, low ghost before high), a ghost's is 0.  Values in
// groups of kPl, as k_planes.
__global__ __launch_bounds__(256) void k_planes_fold(const PlanesArgs a, int g0, int g1, int g2)
{
    const int nx = a.nx, ny = a.ny;
    const unsigned e = blockIdx.x * 256u + threadIdx.x;
    if (e >= (unsigned)nx * (unsigned)ny) return;
    const int y = (int)(e / (unsigned)nx), x = (int)(e - (unsigned)y * (unsigned)nx);
    for (int z = (int)blockIdx.y; z < a.nz; z += (int)gridDim.y) {
        const int g[3] = {g0, g1, g2}, ng[3] = {nx, ny, a.nz}, p[3] = {x, y, z};
        int lo[3], hi[3];  // the low and the high ghost that copy the cell, or -1
        bool inner = true;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const int n = ng[d] - 2 * g[d], i = p[d] - g[d];
            lo[d] = (g[d] > 0 && i >= n - g[d]) ? i - (n - g[d]) : -1;
            hi[d] = (g[d] > 0 && i < g[d]) ? g[d] + n + i : -1;
            inner = inner && i >= 0 && i < n;
        }
        double *s = a.soa + x + (long long)a.sy * y + (long long)a.sz * z;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            if (!a.aos[k]) continue;
            const int nc = a.map[k].nc;
            for (int c0 = 0; c0 < nc; c0 += kPl) {
                double fx[kPl];
#pragma unroll
                for (int c = 0; c < kPl; c++) fx[c] = 0.0;
                if (inner) {
                    for (int i0 = 0; i0 < 3; i0++) {
                        const int cx = i0 == 0 ? x : (i0 == 1 ? lo[0] : hi[0]);
                        if (cx < 0) continue;
                        double fy[kPl];
                        for (int i1 = 0; i1 < 3; i1++) {
                            const int cy = i1 == 0 ? y : (i1 == 1 ? lo[1] : hi[1]);
                            if (cy < 0) continue;
                            double fz[kPl];
                            for (int i2 = 0; i2 < 3; i2++) {
                                const int cz = i2 == 0 ? z : (i2 == 1 ? lo[2] : hi[2]);
                                if (cz < 0) continue;
                                const double *q = a.aos[k] + (cx + (long long)nx * (cy + (long long)ny * cz)) * nc;
                                double v[kPl];
#pragma unroll
                                for (int c = 0; c < kPl; c++) v[c] = q[min(c0 + c, nc - 1)];
#pragma unroll
                                for (int c = 0; c < kPl; c++) fz[c] = i2 == 0 ? v[c] : fz[c] + v[c];
                            }
#pragma unroll
                            for (int c = 0; c < kPl; c++) fy[c] = i1 == 0 ? fz[c] : fy[c] + fz[c];
                        }
#pragma unroll
                        for (int c = 0; c < kPl; c++) fx[c] = i0 == 0 ? fy[c] : fx[c] + fy[c];
                    }
                }
#pragma unroll
                for (int c = 0; c < kPl; c++) {
                    if (c0 + c >= nc) break;
                    s[(long long)a.map[k].planes[c0 + c] * a.sv] = fx[c];
                }
            }
        }
    }
}

// ------------------------------------------------------------ launchers ----

hipError_t launch_dtslots_init(unsigned long long *slots, int nslots, hipStream_t st)
{
    hipLaunchKernelGGL(k_dtslots_init, dim3((unsigned)((nslots + 255) / 256)), dim3(256), 0, st, slots, nslots);
    return hipGetLastError();
}

hipError_t launch_dtslots_final(unsigned long long *slots, int nslots, int nsets, double *out, hipStream_t st)
{
    if (nsets <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_dtslots_final, dim3((unsigned)nsets), dim3(256), 0, st, slots, nslots, out);
    return hipGetLastError();
}

hipError_t launch_dt(const DtArgs &a, double *part, double *out, hipStream_t st)
{
    const long long ncell = (long long)a.n[0] * a.n[1] * a.n[2];
    if (ncell >= (1ll << 32)) return hipErrorInvalidValue;
    long long nb = (ncell + 255) / 256;
    nb = nb > 2048 ? 2048 : nb;
    if (a.magnetized)
        hipLaunchKernelGGL(k_dt_partial<true>, dim3((unsigned)nb), dim3(256), 0, st, a, part);
    else
        hipLaunchKernelGGL(k_dt_partial<false>, dim3((unsigned)nb), dim3(256), 0, st, a, part);
    hipLaunchKernelGGL(k_dt_final, dim3(1), dim3(256), 0, st, part, (int)nb, out);
    return hipGetLastError();
}

hipError_t launch_dt_list(const DtArgs *jobs, int nblocks, int nfl, long long maxcells, unsigned long long *slots,
                          int nslots, int per_block, hipStream_t st)
{
    if (nblocks <= 0) return hipSuccess;
    if (maxcells >= (1ll << 32)) return hipErrorInvalidValue;
    // about 2048 workgroups in all, at most one per 256 cells of the largest block
    const long long njobs = (long long)nblocks * nfl;
    long long per = (2048 + njobs - 1) / njobs, most = (maxcells + 255) / 256;
    per = per > most ? most : per;
    for (long long j0 = 0; j0 < njobs; j0 += 32768 / nfl * nfl) {
        const long long n = njobs - j0 < 32768 / nfl * nfl ? njobs - j0 : 32768 / nfl * nfl;
        hipLaunchKernelGGL(k_dt_list, dim3((unsigned)per, (unsigned)n), dim3(256), 0, st, jobs + j0, nfl,
                           slots + (per_block ? 4ll * nslots * (j0 / nfl) : 0ll), nslots, per_block);
    }
    return hipGetLastError();
}

hipError_t launch_planes(bool in, const PlanesArgs &a, hipStream_t st)
{
    const long long pl = (long long)a.nx * a.ny;
    if (pl > 0xffffff00ll) return hipErrorInvalidValue;  // more cells than memory holds
    const dim3 grid((unsigned)((pl + 255) / 256), (unsigned)(a.nz < 65535 ? a.nz : 65535));
    if (in)
        hipLaunchKernelGGL(k_planes<true>, grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(k_planes<false>, grid, dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_planes_fold(const PlanesArgs &a, const int g[3], hipStream_t st)
{
    const long long pl = (long long)a.nx * a.ny;
    if (pl > 0xffffff00ll) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((pl + 255) / 256), (unsigned)(a.nz < 65535 ? a.nz : 65535));
    hipLaunchKernelGGL(k_planes_fold, grid, dim3(256), 0, st, a, g[0], g[1], g[2]);
    return hipGetLastError();
}

hipError_t launch_fill_periodic(const GhostArgs &a, hipStream_t st)
{
    const long long nx = a.ng[0], ny = a.ng[1], iz = a.n[2];
    const long long total = 2 * a.g[2] * nx * ny + 2 * a.g[1] * iz * nx + 2 * a.g[0] * iz * (long long)a.n[1];
    if (total == 0) return hipSuccess;
    if (total > 0xffffff00ll) return hipErrorInvalidValue;  // more cells than memory holds
    hipLaunchKernelGGL(k_fill_periodic, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_scale(double *x, long long n, double fac, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_scale, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, n, fac);
    return hipGetLastError();
}

hipError_t launch_fill_items(const unsigned *first, int nblocks, unsigned *items, hipStream_t st)
{
    if (nblocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_items, dim3((unsigned)nblocks), dim3(256), 0, st, first, nblocks, items);
    return hipGetLastError();
}

hipError_t launch_exchange_faces(const FaceJob *jobs, const int *wgjob, int nwg, hipStream_t st)
{
    if (nwg <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_exchange_faces, dim3((unsigned)nwg), dim3(256), 0, st, jobs, wgjob);
    return hipGetLastError();
}

hipError_t launch_copy_blocks(const CopyJob *jobs, int njobs, hipStream_t st)
{
    if (njobs <= 0) return hipSuccess;
    const unsigned gy = (unsigned)(njobs < 65535 ? njobs : 65535);
    hipLaunchKernelGGL(k_copy_blocks, dim3(256, gy), dim3(256), 0, st, jobs, njobs);
    return hipGetLastError();
}

hipError_t launch_zero_u32(unsigned *p, int n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_zero_u32, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n);
    return hipGetLastError();
}

}  // namespace pk
