// pk_kernels.hpp -- kernel argument blocks and launchers (host side).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace pk {

// fc_at value of a pencil without that flux point: below every cell a lane
// of a tile can hold (tiles start at most a halo before the pencil).
constexpr int kFcNone = -(1 << 20);

struct SweepArgs {
    const double *src;   // state read with halo (current stage input)
    const double *base;  // U0 of the update (start-of-step state); == src at the first stage
    double *dst;         // output state (never aliases src)
    long long sv;        // plane stride (elements)
    int sy, sz;          // y and z strides (elements), x stride is 1
    int ng[3];           // ghost-padded extents
    int g[3];            // ghost layers per direction (0 where the direction is inactive)
    int n[3];            // interior extents
    int TP, TS;          // tile: TP pencils x TS cells along the sweep
    int chunks;          // tiles along the sweep direction
    int ptiles;          // tiles over the transverse interior, pencils flattened (d1 fastest)
    int out;             // output cells per tile along the sweep (TS-8 fused, TS-4 per stage)
    int lim, limb;       // limiter for fluid primitives / for B and psi
    double gam, gam_1;
    double c1;           // dt/dx coefficient of the (first) stage
    double c2;           // dt/dx coefficient of the second stage (fused mode)
    double ch;           // GLM cleaning speed
    double psi_fac;      // multiplier applied to psi on output (fused GLM damping), else 1
    double smalld, smallei;
    int use_smalld, use_smallei;
    int ei_flag;         // record negative internal energies (disallow_negatives, sources.F90:425)
    unsigned *flags;     // device: bit 0 negative density, bit 1 negative internal energy
    unsigned long long *dmass;  // device: floor-added mass / cell volume, exact counters (pk_mass.hpp)
    // fused mode only:
    int wrap;            // 1: read each ghost position's interior pre-image (a block periodic on itself)
                         // instead of the ghost; no sweep writes ghosts
    unsigned long long *dtslots;  // if set: per slot, min of dl_d/c_d (d = x, y, z) and max c of the
                                  // cells written, as FP64 bit patterns (timestep_fluid of the next step)
    int nslots;
    int has_dir[3];
    double dl[3];
    // stage mode only:
    int gwgs;            // the launch's first gwgs workgroups (a multiple of 8) copy the cells outside the
                         // transverse interior from src to dst (set by the launcher)
    // stage mode only: fine/coarse flux points of the pencils (null when none)
    const int *fc_at;    // [4][fc_npen]: the cell whose right-face flux is replaced (li, ri) or saved (lo, ro);
                         // kFcNone (below every lane's cell) where absent
    const int *fc_slot;  // [4][fc_npen]: the record of each active point in fc_in (li, ri) or fc_out (lo, ro)
    const double *fc_in; // records of fc_rec values: replacement fluxes of the active li, ri points
    double *fc_out;      // records: the saved fluxes of the active lo, ro points
    int fc_npen;         // pencils of the transverse interior (d1 fastest)
    int fc_rec;          // record length: the u-fluxes of every fluid, then [B, psi] with a magnetic field
    int fc_beg;          // this fluid's first u-flux in a record
    int fc_boff;         // first [B, psi] flux in a record
};

struct GhostArgs {
    double *u;
    long long sv;
    int sy, sz;
    int ng[3], g[3], n[3];
    int plane0, nplanes;
};

// Fortran AoS component c of nc <-> device plane planes[c].
struct PlaneMap {
    int nc;
    int planes[16];
};

struct DtArgs {
    const double *u;
    long long sv;
    int sy, sz;
    int ng[3], g[3], n[3];
    int plane0;    // rho plane of the fluid
    int bplane;    // Bx plane (magnetized fluid)
    int magnetized;
    int has_dir[3];
    double dl[3];
    double gam, gam_1;
};

// Per-step scalars of the batched sweep, in device memory so that a captured
// graph replays every step unchanged.
struct StepScalars {
    double dt;       // the step's dt; the sweep forms (rk_coef*dt)/dl per block
    double ch;       // GLM cleaning speed
    double psi_fac;  // GLM damping factor applied by the last sweep of each substep
    double pad;
};

#if defined(__HIPCC__)
// This workgroup's place in an XCD-aware order: workgroup i runs on XCD i % 8,
// so each XCD gets a contiguous range of places, and tiles that share halo
// cells or cache lines share an L2.
__device__ __forceinline__ unsigned xcd_order(unsigned w, unsigned n)
{
    const unsigned full = n / 8u * 8u;
    return w < full ? (w % 8u) * (full / 8u) + w / 8u : w;
}
__device__ __forceinline__ unsigned xcd_order() { return xcd_order(blockIdx.x, gridDim.x); }

// The t-th ghost cell of a block of i (interior) cells and g ghost layers on
// each side per direction: z slabs (whole planes), then y slabs (interior z),
// then x slabs.  False past the last one.
__device__ __forceinline__ bool ghost_cell(unsigned t, const unsigned (&i)[3], const unsigned (&g)[3], unsigned (&c)[3])
{
    const unsigned nx = i[0] + 2u * g[0], ny = i[1] + 2u * g[1];
    const unsigned rz = 2u * g[2] * nx * ny, ry = 2u * g[1] * i[2] * nx, rx = 2u * g[0] * i[2] * i[1];  // < 2^32 (launchers)
    if (t < rz) {
        const unsigned pl = nx * ny, l = t / pl, r = t - l * pl;
        c[2] = l < g[2] ? l : i[2] + l;
        c[1] = r / nx;
        c[0] = r - c[1] * nx;
        return true;
    }
    t -= rz;
    if (t < ry) {
        const unsigned pl = 2u * g[1] * nx, l = t / pl, r = t - l * pl;
        const unsigned q = r / nx;
        c[2] = g[2] + l;
        c[1] = q < g[1] ? q : i[1] + q;
        c[0] = r - q * nx;
        return true;
    }
    t -= ry;
    if (t >= rx) return false;
    const unsigned pl = 2u * g[0] * i[1], l = t / pl, r = t - l * pl;
    const unsigned q = r / (2u * g[0]), e = r - q * 2u * g[0];
    c[2] = g[2] + l;
    c[1] = g[1] + q;
    c[0] = e < g[0] ? e : i[0] + e;
    return true;
}

// Copies of the planes of one cell, G at a time so that the loads of a group
// are in flight together.
template <int G>
__device__ __forceinline__ void copy_planes(const double *s, long long ssv, double *d, long long dsv, int np)
{
    for (int v0 = 0; v0 < np; v0 += G) {
        double x[G];
#pragma unroll
        for (int v = 0; v < G; v++) x[v] = s[(long long)(v0 + v < np ? v0 + v : np - 1) * ssv];
#pragma unroll
        for (int v = 0; v < G; v++)
            if (v0 + v < np) d[(long long)(v0 + v) * dsv] = x[v];
    }
}
#endif

// Most workgroups of one list launch (the runtime takes fewer than 2^32
// lanes); longer lists take several launches.
constexpr unsigned kListPiece = 1u << 22;

// One launch over a block list, an item per workgroup (k_sweep_list,
// k_sweep_adjoint_list; k_stream_list walks a range of items).  Item `item`
// belongs to block items[item] and is that block's tile (or range of its
// stream) item - first[block].  The hardware hands the workgroups out: with
// resident workgroups taking items from a queue, or each walking a fixed range
// of them, a sweep of 12 linked MHD blocks (120x96x80 cells in all) is
// limited by the latency of a workgroup's successive tiles and by the block
// arguments a loop keeps in scalar registers (40 spilled); a step took 935 us
// with queues, 821 with ranges, 727 an item a workgroup (48 blocks of two
// fluids: 3190, 2950, 2427; 20 2-D blocks: 369, 355, 280).
struct ListArgs {
    const SweepArgs *args;   // per block: geometry, pointers (src = buffer 0), tile shape
    const unsigned *first;   // per block: first item (nblocks + 1 entries)
    const unsigned *items;   // per item: block index
    unsigned nitems;
    unsigned item0;          // first item of the launch
    int parity;              // 1: read buffer 1, write buffer 0
    int apply_fac;           // multiply psi by step->psi_fac
    int given;               // 1: the ghosts are read as they are, whatever the blocks' wrap
    const StepScalars *step;      // one for the whole list, or one per block (per_block)
    unsigned long long *dtslots;  // if set: fold timestep_fluid of the cells written into these slots
    int nslots;                   // slots (per block when per_block)
    int per_block;                // independent instances: each block has its own dt, ch, psi factor
                                  // and its own nslots dt slots
    const unsigned *bpos;         // per_block: each block's position among the instances (null: its index)
};

// One device-to-device copy of a batch (k_copy_blocks).
struct CopyJob {
    const double *src;
    double *dst;
    long long n;  // doubles
};

// One face of a ghost exchange (k_exchange_faces): the box ext[0] x ext[1]
// x ext[2] of every plane, from the neighbour's state at sorg to this
// block's at dorg (ghosted coordinates, x fastest; src and dst point at
// cell (0, 0, 0) of plane 0).
struct FaceJob {
    const double *src;
    double *dst;
    long long ssv, dsv;  // plane strides
    int ssy, ssz, dsy, dsz;
    int sorg[3], dorg[3], ext[3];
    int nplanes;
    int wg0;             // the job's first workgroup in its launch (kFaceCells cells each)
};
// Cells one workgroup of k_exchange_faces copies (every plane of each), one per lane.
constexpr int kFaceCells = 256;

// Arrays of the reference layout and the planes of a state (k_planes):
// aos[k] holds map[k].nc components per cell, null: not converted.
struct PlanesArgs {
    double *aos[3];
    PlaneMap map[3];
    double *soa;
    long long sv;
    int nx, ny, nz;  // ghosted extents
    int sy, sz;
};

// The tile of at most nt lanes that needs the fewest workgroups for npen pencils
// of span cells, where a tile of ts cells finishes ts - lost of them: over the
// pencil counts tp, the pencil in equal chunks of the longest tile that fits.  Returns the workgroups.  Along x ties go to the longer tile (fewer
// halo cells read).  Along y and z the lanes of a tile read tp cells in a row,
// so at least 3 pencils are taken and ties go to the longest tile of 4 or more
// (HD 224^3, y, 256 lanes: 4x64 575 us, 2x120 586, 1x232 > 640; HD 96^3, y:
// 4x56 62 us, 2x104 65; MHD 131x98x77, y: 4x57 140 us, 2x106 147).
inline long long even_tile(int span, long long npen, int lost, bool along_x, int nt, int &tp_out, int &ts_out)
{
    long long best = -1;
    tp_out = 1;
    ts_out = lost + 1;
    const int tp0 = along_x || npen < 3 ? 1 : 3;
    for (int tp = tp0; tp <= nt / (lost + 1) && (tp <= npen || tp == tp0); tp++) {
        const int k = (span + nt / tp - lost - 1) / (nt / tp - lost);
        const int out = (span + k - 1) / k;
        const long long wgs = (long long)((span + out - 1) / out) * ((npen + tp - 1) / tp);
        if (best < 0 || wgs < best || (wgs == best && !along_x && tp_out < 4)) {
            best = wgs;
            tp_out = tp;
            ts_out = out + lost;
        }
    }
    return best;
}

// Default tile: 256 lanes (MHD 64^3, z: 256 lanes 47 us, 512 lanes 56; the
// register budget of the kernels holds two or three 4-wave workgroups per CU,
// which hide each other's barriers, but one 8-wave workgroup), fewer where
// that leaves some of the 256 CUs without a workgroup (HD 32^3: 4x40 in 256
// workgroups 12.4 us, 6x40 in 171 13.3; HD 16^3: 2x24 in 128 11.3 us, 10x24 in
// 26 12.3 - 13.5).  Against a fixed 3 x 72, which leaves the last chunk of
// most lengths nearly empty: MHD 131x98x77 206, 179, 212 us along x, y, z there,
// 147, 140, 125 here; HD 96^3 82, 77, 82 there, 65, 62, 65 here.
inline void full_tile(int span, long long npen, int lost, bool along_x, int &tp, int &ts)
{
    for (int nt = 256; nt >= 64; nt -= 64)
        if (even_tile(span, npen, lost, along_x, nt, tp, ts) >= 256) return;
}

hipError_t launch_sweep(int dir, bool mhd, bool fused, const SweepArgs &a, hipStream_t st);
// Workgroup size that selects the stream form of the list sweep
// (k_stream_list: one-wave workgroups, each list item a range of a block's
// stream of a.out positions, a.TP pencils per lane group: 1 along x, 8 along
// y and z).
constexpr int kStreamListNt = 64;
// Pencils per lane group of the list stream along direction d.
constexpr int stream_list_tp(int d) { return d == 0 ? 1 : 8; }
// The stream kernels store a fluid's planes of sv cells through raw buffer
// resources over three planes each, whose byte ranges (24 sv) must stay
// below 2^31.
constexpr bool stream_stores_fit(long long sv) { return sv >= 0 && 24 * sv < (1ll << 31); }
// Batched fused sweep with workgroups of nt lanes: a tile each, or, for the
// stream, grid of them, a range of items each (grid = 0: as many as the device
// holds at once, at most one per item).
hipError_t launch_sweep_list(int dir, bool mhd, int lim, int limb, const ListArgs &L, int nt, int grid,
                             hipStream_t st);
int sweep_list_resident(int dir, bool mhd, int lim, int limb, int nt);
hipError_t launch_fill_items(const unsigned *first, int nblocks, unsigned *items, hipStream_t st);
hipError_t launch_copy_blocks(const CopyJob *jobs, int njobs, hipStream_t st);
// the faces of one exchange: jobs[wgjob[w]] is the job of workgroup w (nwg workgroups)
hipError_t launch_exchange_faces(const FaceJob *jobs, const int *wgjob, int nwg, hipStream_t st);
hipError_t launch_zero_u32(unsigned *p, int n, hipStream_t st);
// every ghost cell of a block periodic on itself, in one launch
hipError_t launch_fill_periodic(const GhostArgs &a, hipStream_t st);
hipError_t launch_scale(double *x, long long n, double fac, hipStream_t st);
// timestep slots: cleared once, and again by each launch_dtslots_final, which
// reduces nsets sets of nslots slots to (min dl_x/c, min dl_y/c, min dl_z/c,
// max c) each, written to device or pinned host memory
hipError_t launch_dtslots_init(unsigned long long *slots, int nslots, hipStream_t st);
hipError_t launch_dtslots_final(unsigned long long *slots, int nslots, int nsets, double *out, hipStream_t st);
hipError_t launch_dt(const DtArgs &a, double *part, double *out, hipStream_t st);
// timestep_fluid of nblocks blocks of nfl fluids (jobs: device table, fluids
// of a block together) into the slots; maxcells: cells of the largest block
hipError_t launch_dt_list(const DtArgs *jobs, int nblocks, int nfl, long long maxcells, unsigned long long *slots,
                          int nslots, int per_block, hipStream_t st);
// reference arrays -> planes (in) or planes -> reference arrays
hipError_t launch_planes(bool in, const PlanesArgs &a, hipStream_t st);
// reference arrays -> planes with the ghosts' values added to the interior
// cells they copy (g: ghost layers) and the ghosts cleared
hipError_t launch_planes_fold(const PlanesArgs &a, const int g[3], hipStream_t st);

}  // namespace pk

namespace pk_fast {
// the sweeps of pk_kernels_fast.hip (FMA contraction, fast division)
hipError_t launch_sweep(int dir, bool mhd, bool fused, const pk::SweepArgs &a, hipStream_t st);
hipError_t launch_sweep_list(int dir, bool mhd, int lim, int limb, const pk::ListArgs &L, int nt, int grid,
                             hipStream_t st);
int sweep_list_resident(int dir, bool mhd, int lim, int limb, int nt);
}  // namespace pk_fast
