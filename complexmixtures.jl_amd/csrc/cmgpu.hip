// cmgpu.hip -- MI355X (gfx950) implementation of the MDDF accumulation of
// ComplexMixtures.jl behind the C ABI of include/cmgpu.h.
//
// Two kernel families, chosen per job:
//
// "tiles" -- one solute molecule of any size (proteins, polymers), solvent
// molecules of up to 64 atoms.  Per batch of frames, on the job's stream:
//   k_radii             solvent molecule radius about its centre, then per-frame
//                       FP32 thresholds (guard band)
//   k_wrap_atoms, k_scan_cells, k_scatter
//                       solute atoms in a fine cell grid (counting sort + scan)
//   k_near_mark         cells within cutoff + radius of some solute atom
//   k_prep_solvent_tiles  centre of every solvent molecule, key when near
//   k_scan_sums, k_scan_rows, k_mol_scatter, k_chunk_table
//                       near molecules sorted by the Hilbert key of their cell
//                       (the real pass; the random passes of a frame together),
//                       cut into chunks of whole molecules, one wavefront each:
//                       fewer near a compact solute, more about an extended one
//   k_fill_real         atoms of the near molecules in sorted order, fixed point
//   k_eval_tiles        per chunk: AABB, solute atoms within reach of it staged
//                       in LDS, distances on the matrix cores (columns: molecules
//                       of three atoms, or atoms), minimum and second smallest per
//                       atom, minimum per molecule, records that FP32 decides into
//                       LDS histograms
//   k_resolve           the other molecules in FP64: 0.2 % of those within the cutoff of
//                       a globule in a cubic cell, 0.7 % in a triclinic one
//   k_bulk_compact      ordered list of bulk molecules (inbulk, src/mddf.jl:55-57)
//   k_place_keys, k_place_near
//                       Philox placement (src/rigid_body.jl:107-137): centres
//                       of all slots, then the full placement of the slots whose
//                       centre is near the solute, in sorted order
//   then sort, chunk, k_eval_tiles and k_resolve again for the random passes.
//
// "mols" -- many solute molecules (self MDDF, small solutes), molecules of up
// to 16 atoms:
//   k_cl_keys, k_cl_scan, k_cl_order
//                       molecule radii, molecules in Hilbert order
//   k_cl_build          tiles of 16 solute rows (1, 4, 8 or 16 a molecule),
//                       clusters of 16 solvent molecules, their boxes
//   k_cl_eval           per cluster: every tile whose box is within the cutoff,
//                       distances on the matrix cores, pairs within the cutoff
//                       queued and counted, what FP32 leaves open in FP64
// Larger molecules, and jobs on a caller's scratch: molecule centres in a cell
// list, one thread per solvent molecule evaluating all atom pairs of close
// molecule pairs (k_radii, k_prep_solute_mols, k_prep_solvent,
// k_eval_mols_real).  Both, for the random passes: k_mols_near (slots near their
// drawn solute molecule), k_eval_mols_rand (their placement and records).
//
// k_flush turns integer hits into FP64 accumulators times the frame weight.
//
// Coordinates that are not numbers (or infinite) take part in no distance: a
// solute atom without a position is in no cell and no tile, a solvent molecule of
// which any atom has none is near nothing (tiles), and its placed copies with it.
//
// Exactness.  Candidate pairs are evaluated in FP32, from fixed-point fractions
// of the cell (tiles: differences are exact) or from coordinates in the frame of
// each molecule's cell (mols).  Per atom (tiles) or molecule pair (mols) the
// kernels keep the best and second-best squared distance; when the gap exceeds
// a guard band that bounds the FP32 error, the FP32 argmin is the FP64 argmin
// and its d^2 decides the bin, in FP64 when the bin edge is within the guard.
// Otherwise every pair near the minimum is recomputed in FP64.  Records,
// indices and bins therefore equal those of an FP64 evaluation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <chrono>
#include <climits>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "cm_math.h"
#include "cmgpu.h"

using ull = unsigned long long;

namespace {

constexpr int BLOCK = 256;
constexpr int MAX_NBINS = 8192;

// ---------------------------------------------------------------------------
// device-side structures
// ---------------------------------------------------------------------------
struct Geo {                 // one frame of a batch
    cm::Cell64 cell;
    float H32[9];
    float Hi32[9];
    double sp[3];            // plane spacings
    int nc[3];
    int ncell;
    uint32_t frame;          // 1-based trajectory frame (keys the random streams)
    float cut2_hi;           // FP32 squared distances above this are beyond the cutoff
    float amb;               // best/second gap below which the FP64 resolve is exhaustive
    float rpre2;             // molecule-centre pre-check radius^2 (mols family)
    unsigned ru_bits, rv_bits;   // molecule radii (float bits, atomicMax)
    int err;                 // geometry the kernels cannot handle
    unsigned voids;          // tiles family: solvent molecules without a position (b_prep_solvent_tiles)
    unsigned radii_done;     // blocks of the radii launch that have reported (the last one runs frame_grid)
    float rstage;            // staging radius around a chunk (cutoff + margin), tiles family
    float rnear;             // near-cell radius around a solute atom (cutoff + radius + margin)
    int kbits;               // bits per dimension of the sort keys of the fine cells
    int ortho;               // diagonal cell matrix: cells are boxes (exact near-cell test)
    double guard;            // bound on |d2(FP32) - d2(FP64)| for pairs up to the cutoff
    float guard_up;          // the same, rounded up
    unsigned rs_bits;        // molecule pairs on the matrix cores: largest radius of an A tile about its centre
    // fixed-point fractional coordinates, 2^fix units per cell
    int fix;
    float Hfix[9];           // lattice vectors per unit (FP32)
    float gd0, gd1, gd2;     // guard of a direct FP32 d2 but for the coordinates' rounding: gd0 + gd1 d + gd2 d2 (with decide32's)
    float rho;               // |error| of an FP32 difference of two fixed-point positions, in 2^-24 of its length
    float guard32;           // guard + (cutoff^2 + guard + 1) 2^-21, rounded up: covers FP32 b -+ guard32 rounding
};

struct KP {                  // job parameters, by value
    int Mu, nu, Mv, nv;
    int self_, iref, nbins, usecutoff;
    double binstep, cutsys, cut2, dbulk;
    float inv_binstep;       // 1 / binstep in FP32 (bin estimates only)
    // FP32 thresholds of the all-FP32 decision (decide32), rounded outward:
    // cutoff^2 down / up, binstep^2 (1 -+ 4e-7) down / up, dbulk^2 (1 -+ 4e-7)
    float c2lo32, c2hi32, bs2m32, bs2p32, db2lo32, db2hi32;
    int K;                   // random passes per frame (n_random_samples, 0 for coordination numbers)
    int kb;                  // bulk lists per frame (1 in the atoms family, K in the mols family)
    uint32_t key0, key1;
    const int *gu_ptr, *gu_idx, *gv_ptr, *gv_idx;
    int cap;                 // cell slots per frame
    int F;                   // frames in the batch
    int64_t Nu, Nv;
    int mpt;                 // molecules per chunk of the real pass (tiles family)
    int mpt_r;               // the same of the random passes
    int mpt_auto;            // chunks may be larger than that, as each launch chooses (b_chunk_table)
    int mol_lane;            // tiles family: 3-atom solvent molecules (their three atoms evaluated together)
    int glds;                // molecule-pair kernels: group counts privatised in LDS
    int gnu, gnv;            // group counts of the solute / solvent side
    int NP;                  // passes per frame, 1 + K (tiles family)
    // The random passes of a frame place molecules around the same solute
    // atoms and only their sums are kept, so they are sorted and evaluated
    // together: NG groups of KM passes (the last one may hold fewer), each one
    // row of slots (pass within the group times Mv plus the molecule).
    int KM, NG;
    int kcap;                // molecule sort keys of the real pass: Hilbert positions of the fine cells
    int ksub;                // bits per dimension the random groups' keys have beyond them
    int kcapr;               // sort keys of a random group: kcap << 3 ksub
    // molecule pairs on the matrix cores: rows per solute molecule in an A
    // tile (0: not used; 1: single atoms on both sides); A tiles, super tiles and B
    // clusters per frame
    int rpm, nT, nS, nB;
    int place_all;           // verification: every slot of a random pass placed (molecule pairs), FP64 positions kept (tiles)
};

// MinimumDistance record as the verification getters return it
// (src/minimum_distances.jl:12-19; 0-based i molecule-local, j global)
struct VRec {
    int within;
    int i;
    int64_t j;
    double d;
    int ref;
    int pad;
    double dref;
};

// one side (0: solute, 1: solvent) of the molecule pairs on the matrix cores:
// M molecules of n atoms in the order of their keys (2^bits cells per dimension)
struct ClSide {
    int M, n, bits;
    int *key, *rank;         // [F][M]
    int* ord;                // [F][M] input index; bit 31: drawn by a random pass
    int *cnt, *start;        // [F][8^bits]
    double* cen;             // [F][M][3] centres as k_cl_keys forms them
};

struct Bufs {
    Geo* geo;
    // cell list
    int* cnt;                // [F][cap+1]
    int* start;              // [F][cap+1]
    float4* tmp4;            // [F][nitems] unsorted entries
    int* tmpcell;            // [F][nitems]
    float4* sorted;          // [F][nitems]
    int nitems;              // atoms (atoms family) or solute molecules (mols family)
    // solute molecules (mols family)
    float4* solw;            // [F][Nu] atoms in the frame of their molecule's cell
    float4* ucen;            // [F][Mu]
    // solvent, real pass
    float4* vw;              // [F][Nv]
    int* vcell;              // [F][Mv]
    float4* vcen;            // [F][Mv]
    // random passes
    double* P;               // [F][K][Nv][3]
    float4* vw_r;            // [F][K][Nv]
    float4* vcen_r;          // [F][K][Mv] slots to evaluate, their centres and numbers (count: slot_counts)
    unsigned char* bflag;    // [F][kb][Mv]
    int* blist;              // [F][kb][Mv]
    int* nbulk;              // [F][kb]
    int* uk;                 // [F][K] drawn solute molecule of each random pass
    int* drawn_ptr;          // [F][Mu+1] CSR: solute molecule -> random passes
    int* drawn_idx;          // [F][K]
    // tiles family: near cells and molecules sorted by cell per (frame, pass)
    unsigned char* near;     // [F][cap]
    unsigned* dfield;        // [2][F][cap] 0xffffffff - bits of the distances from a near cell's centre and
                             // lower corner to the nearest solute atom image nearby (0: none), b_dfield
    // (rows of a frame: the real pass, then the NG random groups; row_base, key_row)
    int* mkey;               // [F][NP][Mv] Hilbert key of the centre's cell, -1 when far
    int* mrank;              // [F][NP][Mv] rank of a near molecule among those of its key (count order)
    int* mcnt;               // [F][kcap | NG x kcapr] molecules per key
    int* mstart;             // the same shape: first sorted position of a non-empty key
    int* msum;               // [F][parts of kcap | NG x parts of kcapr] molecules per part of a row's keys
    int* msorted;            // [F][NP][Mv] slots in key order
    int* nnear;              // [F][1 + NG]
    unsigned* resmask;       // per chunk of a launch: molecules left to the FP64 resolve, one word, two in chunks of
                             // more than 32 (over mkey, whose keys the scatter has read by then)
    int* chunk_base;         // chunk offsets of one launch, [F*rows] total, evaluation chunk counter, [F*rows + MPT_AT]
                             // molecules per chunk
    // molecule pairs on the matrix cores (self: one side)
    ClSide cl[2];
    float* clA;              // [F][nT][4][16] rows of the A tiles: x, y, z, squared norm
    float* clB;              // [F][nB][nv][4][16] columns of the B clusters, per atom
    float4* tinfo;           // [F][nT][3] fixed-point centre and radius, box middle, box half sides
    float4* binfo;           // [F][nB][3] the same of the clusters
    float4* sinfo;           // [F][nS][2] box middle and half sides of the super tiles
    // accumulators
    ull* cnt_md; ull* cnt_rdf; ull* cnt_md_r; ull* cnt_rdf_r;
    ull* cnt_gu; ull* cnt_gv; ull* cnt_gu_r; ull* cnt_gv_r;
    ull* stats;              // [0] exhaustive resolves, [2] geometry error bits of the job's frames
    VRec* vrec;              // verification: [F][NP][Mv] records of every pass (null when off)
};

// Device memory addressed as the global address space.  A pointer read from
// memory (the job table of the multi-job stages) is otherwise a generic one,
// and its loads and stores compile to flat instructions, which wait on the
// scalar-load counter too and take 64-bit VGPR addresses; through these they
// are global ones, and scalar loads where the address is uniform.
template <class T>
using gptr = __attribute__((address_space(1))) T*;
typedef float f4v __attribute__((ext_vector_type(4)));

// a frame's geometry in the constant address space (not written while the
// reading kernel runs): fields read where they are used, by scalar loads
using GeoC = __attribute__((address_space(4))) const Geo;

template <class T>
__device__ __forceinline__ T ldg(const T* p)
{
    return *(gptr<const T>)p;
}

// A frame's geometry by value, read through the constant address space (it
// is not written while the reading kernel runs): uniform addresses give
// scalar loads.  Not a template: the memcpy builtin is not available to the
// device side of function templates.
__device__ __forceinline__ Geo ldc_geo(const Geo* p)
{
    Geo g;
    __builtin_memcpy(&g, (__attribute__((address_space(4))) const Geo*)p, sizeof(Geo));
    return g;
}

// Molecules per chunk of a launch, as b_chunk_table left them: a scalar load, from
// another cache line than the counter that the launch's wavefronts increment.
constexpr int MPT_AT = 64;
__device__ __forceinline__ int chunk_molecules(const KP& P, const Bufs& B, bool random)
{
    if (!P.mpt_auto) return random ? P.mpt_r : P.mpt;
    return *(__attribute__((address_space(4))) const int*)(B.chunk_base + P.F * (random ? P.NG : 1) + MPT_AT);
}

// first entry of a row of the sorted molecules: the real pass or random group grp of frame f
__device__ __forceinline__ int64_t row_base(const KP& P, int f, bool random, int grp)
{
    return ((int64_t)f * P.NP + (random ? 1 + (int64_t)grp * P.KM : 0)) * P.Mv;
}

// slots of a random group (all its passes)
__device__ __forceinline__ int group_slots(const KP& P, int grp)
{
    return min(P.KM, P.K - grp * P.KM) * P.Mv;
}

// first key count of row r of frame f (0: real pass, 1 + grp)
__device__ __forceinline__ int64_t key_row(const KP& P, int f, int r)
{
    const int64_t per = (int64_t)P.kcap + (int64_t)P.NG * P.kcapr;
    return f * per + (r > 0 ? P.kcap + (int64_t)(r - 1) * P.kcapr : 0);
}

// the fixed-point centre of a tile's or cluster's info (uniform: scalar loads)
struct GeoI3 { int x, y, z; };
__device__ __forceinline__ GeoI3 fix_info(const float4* p)
{
    const auto* q = (__attribute__((address_space(4))) const int*)p;
    return {q[0], q[1], q[2]};
}

struct Rec {
    int within;
    int i;
    int64_t j;
    double d;
    int ref;
    double dref;
    int bin;                 // 0-based bin of d when known without d (-1: from d)
    int rbin;                // the same for dref
    int bulk;                // d > dbulk when known without d (-1: from d)
};

__device__ __forceinline__ Rec rec_zero()
{
    Rec r;
    r.within = 0; r.i = -1; r.j = -1; r.d = INFINITY; r.ref = 0; r.dref = INFINITY;
    r.bin = -1; r.rbin = -1; r.bulk = -1;
    return r;
}

// offer a within-cutoff pair to an exact record: ties on d go to the
// smallest (i, j) (update_md, src/minimum_distances.jl:30-39)
__device__ __forceinline__ void rec_offer(Rec& r, int i, int64_t j, double d, bool isref)
{
    if (d < r.d || (d == r.d && (i < r.i || (i == r.i && j < r.j)))) {
        r.within = 1; r.i = i; r.j = j; r.d = d;
    }
    if (isref) { r.ref = 1; r.dref = fmin(r.dref, d); }
}

template <class T>
__device__ __forceinline__ void load3(const T* p, int64_t atom, double& x, double& y, double& z)
{
    x = (double)p[3 * atom]; y = (double)p[3 * atom + 1]; z = (double)p[3 * atom + 2];
}

__device__ __forceinline__ float4 mk4(float x, float y, float z, float w) { return make_float4(x, y, z, w); }

// a fixed-point position (tiles family), kept in the bits of a float4 with w
__device__ __forceinline__ float4 fix4(int x, int y, int z, float w)
{
    return mk4(__int_as_float(x), __int_as_float(y), __int_as_float(z), w);
}

// fixed-point difference to FP32 lengths; general cells sum three products
template <class GEO>
__device__ __forceinline__ void fix_cart(const GEO& g, int dx, int dy, int dz, float& x, float& y, float& z)
{
    const float a = (float)dx, b = (float)dy, c = (float)dz;
    x = g.Hfix[0] * a; y = g.Hfix[4] * b; z = g.Hfix[8] * c;
    if (!g.ortho) {
        x = fmaf(g.Hfix[3], b, fmaf(g.Hfix[6], c, x));
        y = fmaf(g.Hfix[1], a, fmaf(g.Hfix[7], c, y));
        z = fmaf(g.Hfix[2], a, fmaf(g.Hfix[5], b, z));
    }
}

__device__ __forceinline__ void cell_of_frac(const Geo& g, double f0, double f1, double f2, int& cell, int& c0, int& c1,
                                             int& c2)
{
    c0 = (int)(f0 * g.nc[0]); if (c0 >= g.nc[0]) c0 = g.nc[0] - 1; if (c0 < 0) c0 = 0;
    c1 = (int)(f1 * g.nc[1]); if (c1 >= g.nc[1]) c1 = g.nc[1] - 1; if (c1 < 0) c1 = 0;
    c2 = (int)(f2 * g.nc[2]); if (c2 >= g.nc[2]) c2 = g.nc[2] - 1; if (c2 < 0) c2 = 0;
    cell = (c2 * g.nc[1] + c1) * g.nc[0] + c0;
}

__device__ __forceinline__ void cell_of_frac(const Geo& g, double f0, double f1, double f2, int& cell)
{
    int c0, c1, c2;
    cell_of_frac(g, f0, f1, f2, cell, c0, c1, c2);
}

// Sub-cells (2^sub per cell and dimension) of the fractional coordinates
// u01(r0), u01(r1), u01(r2), in integers: r 2^-32 is exact in FP64 and so is
// its product with nc (at most 32 + 21 significant bits), so (int)(u01(r) nc) =
// floor(r nc / 2^32) = (r nc) >> 32, always below nc; the cell of cell_of_frac
// is the sub-cell shifted down by sub.
__device__ __forceinline__ void cell_of_draws(const Geo& g, uint32_t r0, uint32_t r1, uint32_t r2, int sub, int& c0,
                                              int& c1, int& c2)
{
    c0 = (int)(((uint64_t)r0 * ((uint64_t)g.nc[0] << sub)) >> 32);
    c1 = (int)(((uint64_t)r1 * ((uint64_t)g.nc[1] << sub)) >> 32);
    c2 = (int)(((uint64_t)r2 * ((uint64_t)g.nc[2] << sub)) >> 32);
}

// fractional coordinates of a point, the lattice translation n = floor(f)
// that brings it into the cell, and the wrapped fractional part
__device__ __forceinline__ void wrap_point(const Geo& g, double x, double y, double z, double fr[3], double n[3])
{
    const double* Hi = g.cell.Hi;
    double f0 = Hi[0] * x + Hi[3] * y + Hi[6] * z;
    double f1 = Hi[1] * x + Hi[4] * y + Hi[7] * z;
    double f2 = Hi[2] * x + Hi[5] * y + Hi[8] * z;
    n[0] = floor(f0); n[1] = floor(f1); n[2] = floor(f2);
    fr[0] = f0 - n[0]; fr[1] = f1 - n[1]; fr[2] = f2 - n[2];
    for (int k = 0; k < 3; k++) if (fr[k] >= 1.0) { fr[k] = 0.0; n[k] += 1.0; }
}

// whether wrapped coordinates are not numbers (NaN or infinite coordinates
// make them NaN)
__device__ __forceinline__ bool undefined3(const double fr[3]) { return fr[0] != fr[0] || fr[1] != fr[1] || fr[2] != fr[2]; }

// fixed-point position of a point (FP64), not wrapped
__device__ __forceinline__ float4 fix_point(const Geo& g, double x, double y, double z, float w)
{
    const double* Hi = g.cell.Hi;
    const double sc = ldexp(1.0, g.fix);
    return fix4((int)rint((Hi[0] * x + Hi[3] * y + Hi[6] * z) * sc), (int)rint((Hi[1] * x + Hi[4] * y + Hi[7] * z) * sc),
                (int)rint((Hi[2] * x + Hi[5] * y + Hi[8] * z) * sc), w);
}

// Molecule made whole around its first atom (minimum image of every atom
// relative to atom 0); returns the centre of coordinates.
template <class T>
__device__ void mol_centre(const Geo& g, const T* x, int64_t a0, int n, double c[3])
{
    double x0, y0, z0;
    load3(x, a0, x0, y0, z0);
    double sx = 0.0, sy = 0.0, sz = 0.0;
    for (int a = 0; a < n; a++) {
        double xa, ya, za, ox, oy, oz;
        load3(x, a0 + a, xa, ya, za);
        cm::minimage(g.cell, xa - x0, ya - y0, za - z0, &ox, &oy, &oz);
        sx += ox; sy += oy; sz += oz;
    }
    c[0] = x0 + sx / n; c[1] = y0 + sy / n; c[2] = z0 + sz / n;
}

// ---------------------------------------------------------------------------
// radii and grid
// ---------------------------------------------------------------------------
// Radius bound of every molecule about its centre (molecule made whole around
// its first atom), FP32 with a margin that covers the FP32 rounding.
__device__ __forceinline__ void minimage32(const Geo& g, float dx, float dy, float dz, float& ox, float& oy, float& oz)
{
    const float* Hi = g.Hi32;
    const float* H = g.H32;
    float nx = rintf(Hi[0] * dx + Hi[3] * dy + Hi[6] * dz);
    float ny = rintf(Hi[1] * dx + Hi[4] * dy + Hi[7] * dz);
    float nz = rintf(Hi[2] * dx + Hi[5] * dy + Hi[8] * dz);
    ox = dx - (H[0] * nx + H[3] * ny + H[6] * nz);
    oy = dy - (H[1] * nx + H[4] * ny + H[7] * nz);
    oz = dz - (H[2] * nx + H[5] * ny + H[8] * nz);
}

// maximum over the threads of a block (blockDim.x a multiple of 64, at most 1024)
__device__ __forceinline__ float block_max(float x)
{
    __shared__ float part[16];
    for (int o = 32; o >= 1; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, 64));
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) part[w] = x;
    __syncthreads();
    float r = part[0];
    for (int k = 1; k < nw; k++) r = fmaxf(r, part[k]);
    return r;
}

__device__ __forceinline__ double halfulp32(double x)
{
    if (!(x > 1e-30)) return 0x1p-150;
    return ldexp(1.0, ilogb(x) - 24);
}


__device__ void frame_grid(const KP& P, const Bufs& B, int mols_family, int f)
{
    Geo& g = B.geo[f];
    auto radius = [](unsigned* p) { return (double)__uint_as_float(__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)); };
    const double ru = mols_family ? radius(&g.ru_bits) : 0.0, rv = radius(&g.rv_bits);
    if (mols_family) {
        double side = P.cutsys + ru + rv + 1e-3 + 1e-7 * (g.sp[0] + g.sp[1] + g.sp[2]);
        int ncell = 1;
        for (int k = 0; k < 3; k++) {
            int n = (int)floor(g.sp[k] / side);
            g.nc[k] = n < 1 ? 1 : n;
            ncell *= g.nc[k];
            if (!(side < g.sp[k])) g.err = 2;   // image enumeration assumes ru+rv+cutoff < spacing
        }
        if (ncell > P.cap) g.err = 3;
        g.ncell = ncell;
        // the job's error bits (bit 0: molecules too large for the cell, bit 1: grid
        // larger than its allocation), read with the accumulators at the end
        if (g.err) atomicOr(&B.stats[2], g.err == 2 ? 1ull : 2ull);
    }
    const double* H = g.cell.H;
    // Fixed point: positions are fractions of the cell in units of 2^-fix, fix
    // leaving room for atoms a molecule radius outside the cell and for
    // differences of two of them.  A position is off by half a unit per
    // fraction, a difference of two by E per coordinate; the difference is
    // exact in integers, and turning it into a length rounds the conversion,
    // the FP32 lattice vector and the product (a diagonal cell: 3 u), plus the
    // additions over terms of at most kappa times the length in a general one.
    const double smin = fmin(g.sp[0], fmin(g.sp[1], g.sp[2]));
    g.fix = 29 - (int)ceil(log2(1.0 + (fmax(ru, rv) + P.cutsys) / smin));
    double kappa = 0.0, hs = 0.0;
    for (int r = 0; r < 3; r++) {
        kappa = fmax(kappa, fabs(H[r]) / g.sp[0] + fabs(H[3 + r]) / g.sp[1] + fabs(H[6 + r]) / g.sp[2]);
        hs = fmax(hs, fabs(H[r]) + fabs(H[3 + r]) + fabs(H[6 + r]));
    }
    for (int k = 0; k < 9; k++) g.Hfix[k] = (float)ldexp(H[k], -g.fix);
    const double rho = g.ortho ? 3.0 : 5.0 * 1.7320508075688772 * kappa;
    g.rho = (float)(rho * (1.0 + 1e-6));
    const double dmax = P.cutsys + 0.5;
    double E, G;
    if (mols_family) {
        const double xm = hs + fmax(ru, rv) + P.cutsys + 1.0;
        E = 10.0 * halfulp32(2.0 * xm) + 1e-7;
        G = E * (2.0 * 1.7320508075688772 * dmax + 3.0 * E) + 8.0 * 0x1p-24 * dmax * dmax;
    } else {
        E = ldexp(hs, -g.fix) + 1e-9;
        G = E * (2.0 * 1.7320508075688772 * dmax + 3.0 * E) + (2.0 * rho + 4.0) * 0x1p-24 * dmax * dmax;
        g.gd0 = (float)(3.0 * E * E + 1e-9) * (1.0f + 1e-6f);
        g.gd1 = (float)(2.0 * 1.7320508075688772 * E) * (1.0f + 1e-5f);
        g.gd2 = (float)(((2.0 * rho + 4.0) + 4.0) * 0x1p-24) * (1.0f + 1e-5f);
    }
    g.guard = G;
    g.guard_up = nextafterf((float)G, INFINITY);
    g.guard32 = nextafterf((float)(G + (P.cut2 + G + 1.0) * 0x1p-21), INFINITY);
    float hi = (float)(P.cut2 + G);
    g.cut2_hi = nextafterf(hi, INFINITY);
    float ulpc = (float)(halfulp32((double)g.cut2_hi) * 2.0);
    g.amb = nextafterf((float)(2.0 * G) + 8.0f * ulpc, INFINITY);
    float rp = (float)(P.cutsys + ru + rv + 1e-2);
    g.rpre2 = rp * rp;
    g.rstage = (float)(P.cutsys + 20.0 * E + 1e-3);
    g.rnear = (float)(P.cutsys + rv + 20.0 * E + 1e-2 + 1e-6 * (g.sp[0] + g.sp[1] + g.sp[2]));
}

// The end of a block of a radii launch: `blocks` of them report per frame, and
// the last one derives the frame's thresholds (a launch of its own took 3 to 5 us
// of every call).  The blocks run on different XCDs: agent-scope atomics, each
// waited for before the report counts.  (A fence would write the L2 back: with
// one per block the radii of 40,000 molecules, 40 frames took 124 us, not 30.)
__device__ __forceinline__ void radii_report(const KP& P, const Bufs& B, int mols_family, int f, float ru, float rv, int blocks)
{
    if (threadIdx.x != 0) return;
    Geo& g = B.geo[f];
    // (with their results used, the maxima are performed before the count)
    unsigned old = 0;
    if (rv > 0.f) old |= atomicMax(&g.rv_bits, __float_as_uint(rv));
    if (ru > 0.f) old |= atomicMax(&g.ru_bits, __float_as_uint(ru));
    asm volatile("s_waitcnt vmcnt(0)" ::"v"(old) : "memory");
    if (atomicAdd(&g.radii_done, 1u) == (unsigned)blocks - 1u) frame_grid(P, B, mols_family, f);
}

// molecule radii (bound on the distance of an atom from the centre of its
// molecule, with a margin over FP32 rounding); blockIdx.y = frame
template <class T>
__device__ __forceinline__ void b_radii(KP P, Bufs B, const T* xu, const T* xv, int do_solute, int bx_, int nbx_, int by_, int nby_)
{
    const int f = by_;
    Geo& g = B.geo[f];
    const int64_t nmol = (int64_t)P.Mv + (do_solute ? P.Mu : 0);
    float rv = 0.f, ru = 0.f;
    for (int64_t m = bx_ * (int64_t)blockDim.x + threadIdx.x; m < nmol; m += (int64_t)nbx_ * blockDim.x) {
        const bool solv = m < P.Mv;
        const T* x = solv ? xv + (int64_t)f * P.Nv * 3 : xu + (int64_t)f * P.Nu * 3;
        const int n = solv ? P.nv : P.nu;
        const int64_t a0 = solv ? m * P.nv : (m - P.Mv) * P.nu;
        double x0, y0, z0;
        load3(x, a0, x0, y0, z0);
        float sx = 0.f, sy = 0.f, sz = 0.f;
        for (int a = 0; a < n; a++) {
            double xa, ya, za;
            load3(x, a0 + a, xa, ya, za);
            float ox, oy, oz;
            minimage32(g, (float)(xa - x0), (float)(ya - y0), (float)(za - z0), ox, oy, oz);
            sx += ox; sy += oy; sz += oz;
        }
        sx /= n; sy /= n; sz /= n;
        float r2 = 0.f;
        for (int a = 0; a < n; a++) {
            double xa, ya, za;
            load3(x, a0 + a, xa, ya, za);
            float ox, oy, oz;
            minimage32(g, (float)(xa - x0), (float)(ya - y0), (float)(za - z0), ox, oy, oz);
            float dx = ox - sx, dy = oy - sy, dz = oz - sz;
            r2 = fmaxf(r2, dx * dx + dy * dy + dz * dz);
        }
        const float r = sqrtf(r2) * 1.0001f + 1e-3f;
        if (solv) rv = fmaxf(rv, r); else ru = fmaxf(ru, r);
    }
    rv = block_max(rv);
    ru = block_max(ru);
    radii_report(P, B, do_solute, f, ru, rv, nbx_);
}

template <class T>
__global__ void k_radii(KP P, Bufs B, const T* xu, const T* xv, int do_solute)
{
    b_radii<T>(P, B, xu, xv, do_solute, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// ---------------------------------------------------------------------------
// cell list: counting sort by cell
// ---------------------------------------------------------------------------
template <class T>
__device__ __forceinline__ void b_wrap_atoms(KP P, Bufs B, const T* xu, int bx_, int nbx_, int by_, int nby_)
{
    int64_t total = (int64_t)P.F * P.nu;
    for (int64_t it = bx_ * (int64_t)blockDim.x + threadIdx.x; it < total; it += (int64_t)nbx_ * blockDim.x) {
        int f = (int)(it / P.nu);
        int i = (int)(it - (int64_t)f * P.nu);
        const Geo g = ldc_geo(B.geo + f);
        double x, y, z;
        load3(xu + (int64_t)f * P.Nu * 3, i, x, y, z);
        double fr[3], n[3];
        wrap_point(g, x, y, z, fr, n);
        int cell;
        cell_of_frac(g, fr[0], fr[1], fr[2], cell);
        int64_t o = (int64_t)f * B.nitems + i;
        // (an atom with a coordinate that is no number has no fixed-point
        // position and no distance: it stays out of the cells)
        if (undefined3(fr)) {
            B.tmp4[o] = fix4(0, 0, 0, __int_as_float(-1));
            B.tmpcell[o] = -1;
            continue;
        }
        const double sc = ldexp(1.0, g.fix);
        B.tmp4[o] = fix4((int)rint(fr[0] * sc), (int)rint(fr[1] * sc), (int)rint(fr[2] * sc), __int_as_float(i));
        B.tmpcell[o] = cell;
        atomicAdd(&B.cnt[(int64_t)f * (P.cap + 1) + cell], 1);
    }
}

template <class T>
__global__ void k_wrap_atoms(KP P, Bufs B, const T* xu)
{
    b_wrap_atoms<T>(P, B, xu, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// Solute molecules (mols family): made whole, centre wrapped into the cell,
// atoms written in the frame of that cell.
template <class T>
__global__ void k_prep_solute_mols(KP P, Bufs B, const T* xu)
{
    int64_t total = (int64_t)P.F * P.Mu;
    for (int64_t it = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; it < total; it += (int64_t)gridDim.x * blockDim.x) {
        int f = (int)(it / P.Mu);
        int u = (int)(it - (int64_t)f * P.Mu);
        const Geo& g = B.geo[f];
        const T* x = xu + (int64_t)f * P.Nu * 3;
        int64_t a0 = (int64_t)u * P.nu;
        double c[3];
        mol_centre(g, x, a0, P.nu, c);
        double fr[3], n[3];
        wrap_point(g, c[0], c[1], c[2], fr, n);
        int cell;
        cell_of_frac(g, fr[0], fr[1], fr[2], cell);
        const double* H = g.cell.H;
        double tx = H[0] * n[0] + H[3] * n[1] + H[6] * n[2];
        double ty = H[1] * n[0] + H[4] * n[1] + H[7] * n[2];
        double tz = H[2] * n[0] + H[5] * n[1] + H[8] * n[2];
        double x0, y0, z0;
        load3(x, a0, x0, y0, z0);
        for (int a = 0; a < P.nu; a++) {
            double xa, ya, za, ox, oy, oz;
            load3(x, a0 + a, xa, ya, za);
            cm::minimage(g.cell, xa - x0, ya - y0, za - z0, &ox, &oy, &oz);
            B.solw[(int64_t)f * P.Nu + a0 + a] = mk4((float)(x0 + ox - tx), (float)(y0 + oy - ty), (float)(z0 + oz - tz), 0.f);
        }
        float4 cw = mk4((float)(c[0] - tx), (float)(c[1] - ty), (float)(c[2] - tz), __int_as_float(u));
        B.ucen[(int64_t)f * P.Mu + u] = cw;
        int64_t o = (int64_t)f * B.nitems + u;
        B.tmp4[o] = cw;
        B.tmpcell[o] = cell;
        atomicAdd(&B.cnt[(int64_t)f * (P.cap + 1) + cell], 1);
    }
}

// exclusive scan of the cell counts, one block per frame; leaves cnt zeroed
__device__ __forceinline__ void b_scan_cells(KP P, Bufs B, int bx_, int nbx_, int by_, int nby_)
{
    __shared__ int wsum[16];
    __shared__ int carry;
    int f = bx_;
    int ncell = B.geo[f].ncell;
    int* cnt = B.cnt + (int64_t)f * (P.cap + 1);
    int* st = B.start + (int64_t)f * (P.cap + 1);
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int base = 0; base < ncell; base += blockDim.x) {
        int idx = base + threadIdx.x;
        int v = idx < ncell ? cnt[idx] : 0;
        int incl = v;
        for (int o = 1; o < 64; o <<= 1) {
            int t = __shfl_up(incl, o, 64);
            if (lane >= o) incl += t;
        }
        if (lane == 63) wsum[wid] = incl;
        __syncthreads();
        int woff = 0;
        for (int w = 0; w < wid; w++) woff += wsum[w];
        int tot = 0;
        for (int w = 0; w < nw; w++) tot += wsum[w];
        if (idx < ncell) { st[idx] = carry + woff + incl - v; cnt[idx] = 0; }
        __syncthreads();
        if (threadIdx.x == 0) carry += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) st[ncell] = carry;
}

__global__ void __launch_bounds__(1024) k_scan_cells(KP P, Bufs B)
{
    b_scan_cells(P, B, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

__device__ __forceinline__ void b_scatter(KP P, Bufs B, int nper, int bx_, int nbx_, int by_, int nby_)
{
    int64_t total = (int64_t)P.F * nper;
    for (int64_t it = bx_ * (int64_t)blockDim.x + threadIdx.x; it < total; it += (int64_t)nbx_ * blockDim.x) {
        int f = (int)(it / nper);
        int e = (int)(it - (int64_t)f * nper);
        int64_t o = (int64_t)f * B.nitems + e;
        int cell = B.tmpcell[o];
        if (cell < 0) continue;   // no position (b_wrap_atoms)
        int64_t cb = (int64_t)f * (P.cap + 1);
        int pos = B.start[cb + cell] + atomicAdd(&B.cnt[cb + cell], 1);
        B.sorted[(int64_t)f * B.nitems + pos] = B.tmp4[o];
    }
}

__global__ void k_scatter(KP P, Bufs B, int nper)
{
    b_scatter(P, B, nper, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// solvent molecules of the real pass, in the frame of their cell
template <class T>
__global__ void k_prep_solvent(KP P, Bufs B, const T* xv)
{
    int64_t total = (int64_t)P.F * P.Mv;
    for (int64_t it = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; it < total; it += (int64_t)gridDim.x * blockDim.x) {
        int f = (int)(it / P.Mv);
        int v = (int)(it - (int64_t)f * P.Mv);
        const Geo& g = B.geo[f];
        const T* x = xv + (int64_t)f * P.Nv * 3;
        int64_t a0 = (int64_t)v * P.nv;
        double c[3];
        mol_centre(g, x, a0, P.nv, c);
        double fr[3], n[3];
        wrap_point(g, c[0], c[1], c[2], fr, n);
        int cell;
        cell_of_frac(g, fr[0], fr[1], fr[2], cell);
        const double* H = g.cell.H;
        double tx = H[0] * n[0] + H[3] * n[1] + H[6] * n[2];
        double ty = H[1] * n[0] + H[4] * n[1] + H[7] * n[2];
        double tz = H[2] * n[0] + H[5] * n[1] + H[8] * n[2];
        double x0, y0, z0;
        load3(x, a0, x0, y0, z0);
        B.vcell[(int64_t)f * P.Mv + v] = cell;
        if (P.self_) continue;   // the pair kernel reads the solute copies (k_prep_solute_mols)
        for (int a = 0; a < P.nv; a++) {
            double xa, ya, za, ox, oy, oz;
            load3(x, a0 + a, xa, ya, za);
            cm::minimage(g.cell, xa - x0, ya - y0, za - z0, &ox, &oy, &oz);
            B.vw[(int64_t)f * P.Nv + a0 + a] = mk4((float)(x0 + ox - tx), (float)(y0 + oy - ty), (float)(z0 + oz - tz), 0.f);
        }
        B.vcen[(int64_t)f * P.Mv + v] = mk4((float)(c[0] - tx), (float)(c[1] - ty), (float)(c[2] - tz), 0.f);
    }
}

// ---------------------------------------------------------------------------
// histogram updates (update_counters!, src/update_counters.jl:43-88)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void group_hit(ull* gc, int nbins, int b, int64_t atom, const int* ptr, const int* idx, int natomspermol)
{
    if (!ptr) {
        int64_t t = atom % natomspermol;
        atomicAdd(&gc[t * nbins + b], 1ull);
    } else {
        for (int k = ptr[atom]; k < ptr[atom + 1]; k++) atomicAdd(&gc[(int64_t)idx[k] * nbins + b], 1ull);
    }
}

// group_hit where the molecule-local atom is known (no division)
__device__ __forceinline__ void group_hit_local(ull* gc, int nbins, int b, int local, int64_t atom, const int* ptr, const int* idx)
{
    if (!ptr) atomicAdd(&gc[(int64_t)local * nbins + b], 1ull);
    else for (int k = ptr[atom]; k < ptr[atom + 1]; k++) atomicAdd(&gc[(int64_t)idx[k] * nbins + b], 1ull);
}

// bins and the dbulk test of a record from its distances where the fast
// decision did not set them (setbin, src/results.jl:28)
__device__ __forceinline__ void rec_complete(const KP& P, Rec& r)
{
    if (r.within && r.bin < 0) {
        r.bin = (int)cm::setbin(r.d, P.binstep) - 1;
        r.bulk = r.d > P.dbulk ? 1 : 0;
    }
    if (r.ref && r.rbin < 0) r.rbin = (int)cm::setbin(r.dref, P.binstep) - 1;
}

__device__ __forceinline__ void hist_record(const KP& P, unsigned* sh, ull* gu, ull* gv, const Rec& r)
{
    if (!r.within) return;
    int b = r.bin;
    if (b >= P.nbins) return;   // unreachable: d <= cutoff (validated at job creation)
    atomicAdd(&sh[b], 1u);
    group_hit(gu, P.nbins, b, r.i, P.gu_ptr, P.gu_idx, P.nu);
    if (P.self_) group_hit(gu, P.nbins, b, r.j, P.gv_ptr, P.gv_idx, P.nu);
    else group_hit(gv, P.nbins, b, r.j, P.gv_ptr, P.gv_idx, P.nv);
    if (r.ref) {
        const int rb = r.rbin;
        if (rb < P.nbins) atomicAdd(&sh[P.nbins + rb], 1u);
    }
}

// Group counts privatised in LDS (small group arrays): the same updates as
// group_hit into a block-local copy, flushed once per block.
__device__ __forceinline__ void group_hit_lds(unsigned* gc, int nbins, int b, int64_t atom, const int* ptr, const int* idx,
                                              int natomspermol)
{
    if (!ptr) {
        const int64_t t = atom % natomspermol;
        atomicAdd(&gc[t * nbins + b], 1u);
    } else {
        for (int k = ptr[atom]; k < ptr[atom + 1]; k++) atomicAdd(&gc[(int64_t)idx[k] * nbins + b], 1u);
    }
}

// md/rdf into the block histogram sh; groups into LDS (shg) when privatised,
// else straight into the global counters
__device__ __forceinline__ void hist_record_mols(const KP& P, unsigned* sh, unsigned* shg, ull* gu, ull* gv, const Rec& r)
{
    if (!shg) {
        hist_record(P, sh, gu, gv, r);
        return;
    }
    if (!r.within) return;
    const int b = r.bin;
    if (b >= P.nbins) return;
    atomicAdd(&sh[b], 1u);
    unsigned* shu = shg;
    unsigned* shv = shg + (int64_t)P.nbins * P.gnu;
    group_hit_lds(shu, P.nbins, b, r.i, P.gu_ptr, P.gu_idx, P.nu);
    if (P.self_) group_hit_lds(shu, P.nbins, b, r.j, P.gv_ptr, P.gv_idx, P.nu);
    else group_hit_lds(shv, P.nbins, b, r.j, P.gv_ptr, P.gv_idx, P.nv);
    if (r.ref) {
        const int rb = r.rbin;
        if (rb < P.nbins) atomicAdd(&sh[P.nbins + rb], 1u);
    }
}

__device__ __forceinline__ void groups_flush(const KP& P, const unsigned* shg, ull* gu, ull* gv)
{
    __syncthreads();
    const int nu_ = P.gnu * P.nbins, nv_ = P.self_ ? 0 : P.gnv * P.nbins;
    for (int k = threadIdx.x; k < nu_; k += blockDim.x)
        if (shg[k]) atomicAdd(&gu[k], (ull)shg[k]);
    for (int k = threadIdx.x; k < nv_; k += blockDim.x)
        if (shg[nu_ + k]) atomicAdd(&gv[k], (ull)shg[nu_ + k]);
}

__device__ __forceinline__ void hist_clear(unsigned* sh, int n)
{
    for (int k = threadIdx.x; k < n; k += blockDim.x) sh[k] = 0u;
    __syncthreads();
}

__device__ __forceinline__ void hist_flush(unsigned* sh, int nbins, ull* md, ull* rdf)
{
    __syncthreads();
    for (int k = threadIdx.x; k < nbins; k += blockDim.x) {
        if (sh[k]) atomicAdd(&md[k], (ull)sh[k]);
        if (sh[nbins + k]) atomicAdd(&rdf[k], (ull)sh[nbins + k]);
    }
}

__device__ __forceinline__ bool inbulk(const KP& P, const Rec& r)
{
    return P.usecutoff ? (r.within && r.bulk == 1) : !r.within;
}

// A record from the FP32 minimum b of a unique argmin, without the FP64
// recompute, when every FP64 d2 in [b - G, b + G] gives the same cutoff test,
// bin and dbulk test.  The bin of d2 is max(1, ceil(fl(sqrt(d2)) / binstep));
// between ((k-1) binstep)^2 (1 + 1e-12) and (k binstep)^2 (1 - 1e-12) it is k
// whatever the FP64 rounding of the square root and the quotient (below 1e-15
// relative), and likewise d > dbulk is decided outside dbulk^2 (1 -+ 1e-12).
// All in FP32 and branch-free: [lo, hi] = b -+ guard32 (guard32 covers the
// FP32 rounding of both sums, so [lo, hi] contains [b - G, b + G]), and every
// threshold is rounded outward: the cutoff^2 bounds, k^2 binstep^2 (1 - 4e-7)
// <= (k binstep)^2 (1 - 1e-12) and (k-1)^2 binstep^2 (1 + 4e-7) >= ((k-1)
// binstep)^2 (1 + 1e-12) after the FP32 roundings of k^2 and the products
// (each below 1.2e-7 relative), and the dbulk^2 bounds likewise.  The bin
// estimate k comes from the hardware square root; any k is safe, the edge
// tests accept it only when it is the bin of every d2 in [lo, hi].  Returns 1
// when no pair can be within the cutoff, 2 when the record is within with the
// 0-based bin and the dbulk flag set, 0 when the interval straddles a decision.
__device__ __forceinline__ int decide32(const KP& P, float G32, float b, int& bin, int& bulk)
{
    const float lo = b - G32, hi = b + G32;
    const int k = max((int)ceilf(__builtin_amdgcn_sqrtf(b) * P.inv_binstep), 1);
    const float kf = (float)k, km = kf - 1.0f;
    const bool inbin = hi < kf * kf * P.bs2m32 && (k == 1 || lo > km * km * P.bs2p32);
    const bool b1 = lo > P.db2hi32, b0 = hi < P.db2lo32;
    const bool okbulk = !P.usecutoff || b1 || b0;
    bin = k - 1;
    bulk = (P.usecutoff && b1) ? 1 : 0;
    const bool within = hi <= P.c2lo32 && inbin && okbulk;
    return lo > P.c2hi32 ? 1 : (within ? 2 : 0);
}

// FP32 running minimum with second best
struct Best {
    float best, second;
    int bi, ba;
    __device__ __forceinline__ void init() { best = INFINITY; second = INFINITY; bi = -1; ba = -1; }
    // branch-free: second smallest = median of (best, second, d2) while
    // best <= second; selects rather than a branch keep the loop straight
    __device__ __forceinline__ void offer(float d2, int i, int a)
    {
        const bool lt = d2 < best;
        second = __builtin_amdgcn_fmed3f(best, second, d2);
        best = lt ? d2 : best;
        bi = lt ? i : bi;
        ba = lt ? a : ba;
    }
};

// neighbour cell (with its lattice shift) of cell c at offset o in one dimension
__device__ __forceinline__ int nb_cell(int c, int o, int n, int& m)
{
    int t = c + o;
    m = t < 0 ? -1 : (t >= n ? 1 : 0);
    return t - m * n;
}

// Wavefront scans and reductions with DPP row shifts and row broadcasts
// (row_shr:1,2,4,8 within rows of 16 lanes, then row_bcast:15 into rows 1
// and 3 and row_bcast:31 into rows 2 and 3); lanes without a source read the
// identity.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_i(int identity, int x)
{
    return __builtin_amdgcn_update_dpp(identity, x, CTRL, ROWS, 0xf, false);
}

__device__ __forceinline__ int wave_incl_scan(int v)
{
    v += dpp_i<0x111, 0xf>(0, v);
    v += dpp_i<0x112, 0xf>(0, v);
    v += dpp_i<0x114, 0xf>(0, v);
    v += dpp_i<0x118, 0xf>(0, v);
    v += dpp_i<0x142, 0xa>(0, v);
    v += dpp_i<0x143, 0xc>(0, v);
    return v;
}

__device__ __forceinline__ float fmin_sel(float a, float b) { return b < a ? b : a; }
__device__ __forceinline__ float fmax_sel(float a, float b) { return b > a ? b : a; }

// a wave-uniform float moved to a scalar register
__device__ __forceinline__ float sgpr_f(float x)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// minimum / maximum over the wavefront, the same in every lane
__device__ __forceinline__ float wave_min(float x)
{
    const int id = __float_as_int(INFINITY);
    x = fmin_sel(x, __int_as_float(dpp_i<0x111, 0xf>(id, __float_as_int(x))));
    x = fmin_sel(x, __int_as_float(dpp_i<0x112, 0xf>(id, __float_as_int(x))));
    x = fmin_sel(x, __int_as_float(dpp_i<0x114, 0xf>(id, __float_as_int(x))));
    x = fmin_sel(x, __int_as_float(dpp_i<0x118, 0xf>(id, __float_as_int(x))));
    x = fmin_sel(x, __int_as_float(dpp_i<0x142, 0xa>(id, __float_as_int(x))));
    x = fmin_sel(x, __int_as_float(dpp_i<0x143, 0xc>(id, __float_as_int(x))));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
__device__ __forceinline__ float wave_max(float x)
{
    const int id = __float_as_int(-INFINITY);
    x = fmax_sel(x, __int_as_float(dpp_i<0x111, 0xf>(id, __float_as_int(x))));
    x = fmax_sel(x, __int_as_float(dpp_i<0x112, 0xf>(id, __float_as_int(x))));
    x = fmax_sel(x, __int_as_float(dpp_i<0x114, 0xf>(id, __float_as_int(x))));
    x = fmax_sel(x, __int_as_float(dpp_i<0x118, 0xf>(id, __float_as_int(x))));
    x = fmax_sel(x, __int_as_float(dpp_i<0x142, 0xa>(id, __float_as_int(x))));
    x = fmax_sel(x, __int_as_float(dpp_i<0x143, 0xc>(id, __float_as_int(x))));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// The frame fields the pair kernels read on every pair, copied into registers
// once: read through the Geo reference they would be reloaded from memory after
// every global store or atomic (which may alias the geometry array).
struct GeoHot {
    float H32[9];
    float cut2_hi, amb, rpre2, guard32;
    double guard;
    int nc[3];
    __device__ explicit GeoHot(const Geo& g)
        : cut2_hi(g.cut2_hi), amb(g.amb), rpre2(g.rpre2), guard32(g.guard32), guard(g.guard)
    {
#pragma unroll
        for (int k = 0; k < 9; k++) H32[k] = g.H32[k];
        nc[0] = g.nc[0]; nc[1] = g.nc[1]; nc[2] = g.nc[2];
    }
};

template <class GEO>
__device__ __forceinline__ void shift_of(const GEO& g, int mx, int my, int mz, float& tx, float& ty, float& tz)
{
    float fx = (float)mx, fy = (float)my, fz = (float)mz;
    tx = g.H32[0] * fx + g.H32[3] * fy + g.H32[6] * fz;
    ty = g.H32[1] * fx + g.H32[4] * fy + g.H32[7] * fz;
    tz = g.H32[2] * fx + g.H32[5] * fy + g.H32[8] * fz;
}

// ---------------------------------------------------------------------------
// minimum distances, mols family (many solute molecules)
// ---------------------------------------------------------------------------
// FP32 evaluation of all atom pairs of solute molecule u (atoms xs) and the
// solvent molecule whose atoms are yw, the solute shifted by t.
__device__ __forceinline__ void pairs_mol(const KP& P, const float4* xs, const float4* yw, float tx, float ty, float tz,
                                          Best& bm, Best& br)
{
    for (int a = 0; a < P.nv; a++) {
        float4 y = yw[a];
        float yx = y.x - tx, yy = y.y - ty, yz = y.z - tz;
        bool isref = (a == P.iref);
        for (int i = 0; i < P.nu; i++) {
            float4 s = xs[i];
            float dx = yx - s.x, dy = yy - s.y, dz = yz - s.z;
            float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
            bm.offer(d2, i, a);
            if (isref) br.offer(d2, i, a);
        }
    }
}

// exact record of the molecule pair (u, v) from the FP32 bests
template <class TU, class YS>
__device__ Rec resolve_mols(const KP& P, const Geo& g, const TU* xuf, int u, int v, YS ysrc, const Best& bm, const Best& br,
                            ull* stats)
{
    Rec r = rec_zero();
    bool exhaustive = false;
    int64_t ibase = (int64_t)u * P.nu, jbase = (int64_t)v * P.nv;
    if (bm.best <= g.cut2_hi) {
        if (bm.second - bm.best > g.amb) {
            int bn, bk;
            const int dd = decide32(P, g.guard32, bm.best, bn, bk);
            if (dd != 0) {
                if (dd == 2) { r.within = 1; r.i = bm.bi; r.j = jbase + bm.ba; r.d = bm.best; r.bin = bn; r.bulk = bk; }
            } else {
                double x0, x1, x2, y0, y1, y2;
                load3(xuf, ibase + bm.bi, x0, x1, x2);
                ysrc(bm.ba, y0, y1, y2);
                double d2 = cm::canon_d2(g.cell, x0, x1, x2, y0, y1, y2);
                if (d2 <= P.cut2) { r.within = 1; r.i = bm.bi; r.j = jbase + bm.ba; r.d = sqrt(d2); }
            }
        } else exhaustive = true;
    }
    if (br.best <= g.cut2_hi) {
        if (br.second - br.best > g.amb) {
            int bn, bk;
            const int dd = decide32(P, g.guard32, br.best, bn, bk);
            if (dd != 0) {
                if (dd == 2) { r.ref = 1; r.dref = br.best; r.rbin = bn; }
            } else {
                double x0, x1, x2, y0, y1, y2;
                load3(xuf, ibase + br.bi, x0, x1, x2);
                ysrc(P.iref, y0, y1, y2);
                double d2 = cm::canon_d2(g.cell, x0, x1, x2, y0, y1, y2);
                if (d2 <= P.cut2) { r.ref = 1; r.dref = sqrt(d2); }
            }
        } else exhaustive = true;
    }
    if (exhaustive) {
        atomicAdd(stats, 1ull);
        r = rec_zero();
        for (int a = 0; a < P.nv; a++) {
            double y0, y1, y2;
            ysrc(a, y0, y1, y2);
            for (int i = 0; i < P.nu; i++) {
                double x0, x1, x2;
                load3(xuf, ibase + i, x0, x1, x2);
                double d2 = cm::canon_d2(g.cell, x0, x1, x2, y0, y1, y2);
                if (d2 <= P.cut2) rec_offer(r, i, jbase + a, sqrt(d2), a == P.iref);
            }
        }
    }
    rec_complete(P, r);
    return r;
}

// LDS pair queue of the molecule-pair kernel: entries per wavefront
constexpr int QCAP = 128;
constexpr int DCAP = 128;   // deferred FP64 entries per wavefront (self)
constexpr int GLDS_MAX = 32 * 1024;   // bytes of LDS group counts per block
constexpr int GLDS_MAX_CL = 64 << 10;   // the same of the molecule pairs on the matrix cores

__device__ __forceinline__ int wave_max_i(int x)
{
    x = max(x, dpp_i<0x111, 0xf>(INT_MIN, x));
    x = max(x, dpp_i<0x112, 0xf>(INT_MIN, x));
    x = max(x, dpp_i<0x114, 0xf>(INT_MIN, x));
    x = max(x, dpp_i<0x118, 0xf>(INT_MIN, x));
    x = max(x, dpp_i<0x142, 0xa>(INT_MIN, x));
    x = max(x, dpp_i<0x143, 0xc>(INT_MIN, x));
    return __builtin_amdgcn_readlane(x, 63);
}

// Lattice shifts m (per dimension, at most three) that map the cell index cv
// of one molecule onto the neighbour cell cu of another, for the offsets o in
// {-1, 0, 1} with wrap(cv + o) == cu, as a set: bit m + 1.  With three or
// more cells per dimension there is exactly one; small grids map several
// offsets onto one cell.  (A bit set rather than an array: dynamically
// indexed arrays live in scratch memory.)
__device__ __forceinline__ int shifts_onto(int cv, int cu, int n)
{
    int set = 0;
    for (int o = -1; o <= 1; o++) {
        int mm;
        if (nb_cell(cv, o, n, mm) == cu) set |= 1 << (mm + 1);
    }
    return set;
}

// the k-th (from 0, ascending) lattice shift of a shift set
__device__ __forceinline__ int nth_shift(int set, int k)
{
    if (k > 0) set &= set - 1;
    if (k > 1) set &= set - 1;
    return __builtin_ctz((unsigned)set) - 1;
}

// Per-frame state of the molecule-pair kernels: records of molecule pairs
// from their FP32 bests (resolve, histograms, bulk flags) and the evaluation
// of one queued pair.
template <class TU, class TV, int NU>
struct PairCtx {
    const KP& P;
    const Bufs& B;
    const Geo& g;
    const GeoHot gh;
    int f;
    const float4* solw;
    const float4* vwf;
    const float4* vcen;
    const int* vcellf;
    const TU* xuf;
    const TV* xvf;
    const int* dp;
    const int* di;
    unsigned* sh;
    unsigned* shg;

    __device__ PairCtx(const KP& P_, const Bufs& B_, int f_, const TU* xu, const TV* xv, unsigned* sh_, unsigned* shg_)
        : P(P_), B(B_), g(B_.geo[f_]), gh(B_.geo[f_]), f(f_), solw(B_.solw + (int64_t)f_ * P_.Nu),
          // self: the solvent side reads the solute copies (the same molecules,
          // wrapped identically), which halves the data each frame touches
          vwf(P_.self_ ? B_.solw + (int64_t)f_ * P_.Nu : B_.vw + (int64_t)f_ * P_.Nv),
          vcen(P_.self_ ? B_.ucen + (int64_t)f_ * P_.Mu : B_.vcen + (int64_t)f_ * P_.Mv), vcellf(B_.vcell + (int64_t)f_ * P_.Mv), xuf(xu + (int64_t)f_ * P_.Nu * 3),
          xvf(xv + (int64_t)f_ * P_.Nv * 3), dp(B_.drawn_ptr + (int64_t)f_ * (P_.Mu + 1)), di(B_.drawn_idx + (int64_t)f_ * P_.K),
          sh(sh_), shg(shg_) {}

    // record of solute molecule uu and solvent molecule vv
    __device__ void emit(int uu, int vv, const Best& bm, const Best& br) const
    {
        const int64_t jb = (int64_t)vv * P.nv;
        const TV* xv = xvf;
        auto ysrc = [&](int a, double& y0, double& y1, double& y2) { load3(xv, jb + a, y0, y1, y2); };
        Rec r = resolve_mols(P, g, xuf, uu, vv, ysrc, bm, br, &B.stats[0]);
        hist_record_mols(P, sh, shg, B.cnt_gu, B.cnt_gv, r);
        if (P.K > 0 && r.within)
            for (int qq = dp[uu]; qq < dp[uu + 1]; qq++)
                B.bflag[((int64_t)f * P.kb + di[qq]) * P.Mv + vv] = inbulk(P, r) ? 1 : 0;
    }

    // md (+2), group and dbulk-flag updates of both orientations of the self
    // pair {u, v} whose minimum distance joins atom bi of u and atom ba of v,
    // in 0-based bin mbin (mbulk: d > dbulk)
    __device__ void self_main(int u, int v, int bi, int ba, int mbin, int mbulk) const
    {
        if (mbin >= P.nbins) return;   // unreachable: d <= cutoff
        atomicAdd(&sh[mbin], 2u);
        if (!P.gu_ptr && !P.gv_ptr) {
            if (shg) {
                atomicAdd(&shg[(int64_t)bi * P.nbins + mbin], 2u);
                atomicAdd(&shg[(int64_t)ba * P.nbins + mbin], 2u);
            } else {
                atomicAdd(&B.cnt_gu[(int64_t)bi * P.nbins + mbin], 2ull);
                atomicAdd(&B.cnt_gu[(int64_t)ba * P.nbins + mbin], 2ull);
            }
        } else {
            // custom groups: the solute side is looked up with the
            // molecule-local index, the solvent side with the global one
            const int64_t ju = (int64_t)u * P.nv + bi, jv = (int64_t)v * P.nv + ba;
            if (shg) {
                group_hit_lds(shg, P.nbins, mbin, bi, P.gu_ptr, P.gu_idx, P.nu);
                group_hit_lds(shg, P.nbins, mbin, jv, P.gv_ptr, P.gv_idx, P.nu);
                group_hit_lds(shg, P.nbins, mbin, ba, P.gu_ptr, P.gu_idx, P.nu);
                group_hit_lds(shg, P.nbins, mbin, ju, P.gv_ptr, P.gv_idx, P.nu);
            } else {
                group_hit(B.cnt_gu, P.nbins, mbin, bi, P.gu_ptr, P.gu_idx, P.nu);
                group_hit(B.cnt_gu, P.nbins, mbin, jv, P.gv_ptr, P.gv_idx, P.nu);
                group_hit(B.cnt_gu, P.nbins, mbin, ba, P.gu_ptr, P.gu_idx, P.nu);
                group_hit(B.cnt_gu, P.nbins, mbin, ju, P.gv_ptr, P.gv_idx, P.nu);
            }
        }
        if (P.K > 0) {
            const int bulk = P.usecutoff ? mbulk : 0;
            for (int qq = dp[u]; qq < dp[u + 1]; qq++) B.bflag[((int64_t)f * P.kb + di[qq]) * P.Mv + v] = bulk;
            for (int qq = dp[v]; qq < dp[v + 1]; qq++) B.bflag[((int64_t)f * P.kb + di[qq]) * P.Mv + u] = bulk;
        }
    }

    // the same of solute molecule u and solvent molecule v (cross)
    __device__ void cross_main(int u, int v, int i, int a, int mbin, int mbulk) const
    {
        if (mbin >= P.nbins) return;   // unreachable: d <= cutoff
        atomicAdd(&sh[mbin], 1u);
        const int64_t j = (int64_t)v * P.nv + a;
        if (shg) {
            unsigned* shv = shg + (int64_t)P.nbins * P.gnu;
            if (!P.gu_ptr) atomicAdd(&shg[(int64_t)i * P.nbins + mbin], 1u);
            else group_hit_lds(shg, P.nbins, mbin, i, P.gu_ptr, P.gu_idx, P.nu);
            if (!P.gv_ptr) atomicAdd(&shv[(int64_t)a * P.nbins + mbin], 1u);
            else group_hit_lds(shv, P.nbins, mbin, j, P.gv_ptr, P.gv_idx, P.nv);
        } else {
            group_hit_local(B.cnt_gu, P.nbins, mbin, i, i, P.gu_ptr, P.gu_idx);
            group_hit_local(B.cnt_gv, P.nbins, mbin, a, j, P.gv_ptr, P.gv_idx);
        }
        if (P.K > 0) {
            const int bulk = P.usecutoff ? mbulk : 0;
            for (int qq = dp[u]; qq < dp[u + 1]; qq++) B.bflag[((int64_t)f * P.kb + di[qq]) * P.Mv + v] = bulk;
        }
    }

    __device__ void rdf_hit(int bin) const
    {
        if (bin < P.nbins) atomicAdd(&sh[P.nbins + bin], 1u);
    }

    // Self mode, FP32 stage of the unordered pair {u, v}: both orientations
    // share the distance, the atom pair and the bins of the minimum (the FP64
    // distance is symmetric: the minimum image of -delta is the negated one,
    // rounding included), so md and default groups get +2 in one update; the
    // reference-atom parts belong to their orientation (a reference distance
    // is never below the minimum, so its count needs no test of the main
    // part).  Parts the FP32 interval cannot decide are returned as a mask
    // for the deferred FP64 stage: 1 the minimum, 2 the reference atom of v,
    // 4 the reference atom of u, 8 the whole pair exhaustively (an argmin
    // that FP32 cannot separate).  d0, d1 carry the pair and its argmins.
    __device__ int emit_self(int u, int v, const Best& bm, const Best& brv, const Best& bru, int4& d0, int4& d1) const
    {
        d0 = make_int4(u, v, bm.bi, bm.ba);
        d1 = make_int4(brv.bi, bru.bi, 0, 0);
        const bool amb = (bm.best <= gh.cut2_hi && !(bm.second - bm.best > gh.amb)) ||
                         (brv.best <= gh.cut2_hi && !(brv.second - brv.best > gh.amb)) ||
                         (bru.best <= gh.cut2_hi && !(bru.second - bru.best > gh.amb));
        if (amb) return 8;
        int bm_bin, bm_bulk, rv_bin, ru_bin, dummy;
        const int dmain = bm.best <= gh.cut2_hi ? decide32(P, gh.guard32, bm.best, bm_bin, bm_bulk) : 1;
        const int drv = brv.best <= gh.cut2_hi ? decide32(P, gh.guard32, brv.best, rv_bin, dummy) : 1;
        const int dru = bru.best <= gh.cut2_hi ? decide32(P, gh.guard32, bru.best, ru_bin, dummy) : 1;
        if (dmain == 2) self_main(u, v, bm.bi, bm.ba, bm_bin, bm_bulk);
        if (drv == 2) rdf_hit(rv_bin);
        if (dru == 2) rdf_hit(ru_bin);
        return (dmain == 0 ? 1 : 0) | (drv == 0 ? 2 : 0) | (dru == 0 ? 4 : 0);
    }

    // Self mode, deferred FP64 stage of one pair (mask and entry from
    // emit_self).  The three distances are formed together so their loads
    // are in flight at once; parts outside the mask are discarded.
    __device__ void self_deferred(int4 d0, int4 d1, int mask) const
    {
        const int u = d0.x, v = d0.y;
        if (mask & 8) {
            atomicAdd(&B.stats[0], 2ull);
            self_exhaustive(u, v);
            return;
        }
        const int64_t ub = (int64_t)u * P.nu, vb = (int64_t)v * P.nv;
        double a0, a1, a2, b0, b1, b2, c0, c1, c2, e0, e1, e2, p0, p1, p2, q0, q1, q2;
        load3(xuf, ub + max(d0.z, 0), a0, a1, a2);
        load3(xvf, vb + max(d0.w, 0), b0, b1, b2);
        load3(xuf, ub + max(d1.x, 0), c0, c1, c2);
        load3(xvf, vb + P.iref, e0, e1, e2);
        load3(xuf, (int64_t)v * P.nu + max(d1.y, 0), p0, p1, p2);
        load3(xvf, (int64_t)u * P.nv + P.iref, q0, q1, q2);
        const double dm = cm::canon_d2(g.cell, a0, a1, a2, b0, b1, b2);
        const double dr = cm::canon_d2(g.cell, c0, c1, c2, e0, e1, e2);   // atoms of u vs the reference atom of v
        const double du = cm::canon_d2(g.cell, p0, p1, p2, q0, q1, q2);   // atoms of v vs the reference atom of u
        if ((mask & 1) && dm <= P.cut2) {
            const double d = sqrt(dm);
            self_main(u, v, d0.z, d0.w, (int)cm::setbin(d, P.binstep) - 1, d > P.dbulk ? 1 : 0);
        }
        if ((mask & 2) && dr <= P.cut2) rdf_hit((int)cm::setbin(sqrt(dr), P.binstep) - 1);
        if ((mask & 4) && du <= P.cut2) rdf_hit((int)cm::setbin(sqrt(du), P.binstep) - 1);
    }

    // both orientations of a self pair from one set of FP64 distances: the
    // records of (u, v) and (v, u) with their own tie order (update_md,
    // src/minimum_distances.jl:30-39) and reference atoms
    __device__ void self_exhaustive(int u, int v) const
    {
        Rec r1 = rec_zero(), r2 = rec_zero();
        const int64_t ub = (int64_t)u * P.nu, vb = (int64_t)v * P.nv;
        const int n = NU > 0 ? NU : P.nu;
        auto offer = [&](int i, int a, double x0, double x1, double x2, double y0, double y1, double y2) {
            const double d2 = cm::canon_d2(g.cell, x0, x1, x2, y0, y1, y2);
            if (d2 <= P.cut2) {
                const double d = sqrt(d2);
                rec_offer(r1, i, vb + a, d, a == P.iref);
                rec_offer(r2, a, ub + i, d, i == P.iref);
            }
        };
#pragma unroll 1
        for (int a = 0; a < n; a++) {
            double y0, y1, y2;
            load3(xvf, vb + a, y0, y1, y2);
            if constexpr (NU > 0 && NU <= 4) {
#pragma unroll
                for (int i = 0; i < NU; i++) {
                    double x0, x1, x2;
                    load3(xuf, ub + i, x0, x1, x2);
                    offer(i, a, x0, x1, x2, y0, y1, y2);
                }
            } else {
#pragma unroll 1
                for (int i = 0; i < n; i++) {
                    double x0, x1, x2;
                    load3(xuf, ub + i, x0, x1, x2);
                    offer(i, a, x0, x1, x2, y0, y1, y2);
                }
            }
        }
        exact_record(u, v, r1);
        exact_record(v, u, r2);
    }

    // counts and dbulk flags of the FP64 record of solvent molecule v about u
    __device__ void exact_record(int u, int v, Rec r) const
    {
        rec_complete(P, r);
        hist_record_mols(P, sh, shg, B.cnt_gu, B.cnt_gv, r);
        if (P.K > 0 && r.within)
            for (int qq = dp[u]; qq < dp[u + 1]; qq++)
                B.bflag[((int64_t)f * P.kb + di[qq]) * P.Mv + v] = inbulk(P, r) ? 1 : 0;
    }

    // one queued pair {u, v, cell of u, shift code or -1}: every shift of the
    // pair, both orientations in self mode
    __device__ int eval_pair(int4 e, int4& d0, int4& d1) const
    {
        const int u = e.x, v = e.y, cu = e.z;
        const int nc0 = gh.nc[0], nc1 = gh.nc[1], nc2 = gh.nc[2];
        int mxs, mys, mzs;   // shift sets (bit m + 1)
        if (e.w >= 0) {
            mxs = 1 << (e.w % 3);
            mys = 1 << ((e.w / 3) % 3);
            mzs = 1 << (e.w / 9);
        } else {
            const int vc = vcellf[v];
            mxs = shifts_onto(vc % nc0, cu % nc0, nc0);
            mys = shifts_onto((vc / nc0) % nc1, (cu / nc0) % nc1, nc1);
            mzs = shifts_onto(vc / (nc0 * nc1), cu / (nc0 * nc1), nc2);
        }
        const int kx = __popc(mxs), ky = __popc(mys), kz = __popc(mzs);
        const float4* xs = solw + (int64_t)u * P.nu;
        const float4* yw = vwf + (int64_t)v * P.nv;
        const float4 cv = vcen[v];
        const float4 cuc = B.ucen[(int64_t)f * P.Mu + u];
        Best bm, brv, bru;
        bm.init(); brv.init(); bru.init();
        if constexpr (NU > 0) {
            // self with NU-atom molecules: both molecules in registers, all
            // loads in flight together
            float4 X[NU], Y[NU];
#pragma unroll
            for (int i = 0; i < NU; i++) X[i] = xs[i];
#pragma unroll
            for (int a = 0; a < NU; a++) Y[a] = yw[a];
            if constexpr (NU <= 4) {
                auto atoms = [&](float tx, float ty, float tz) {
#pragma unroll
                    for (int a = 0; a < NU; a++) {
                        const float yx = Y[a].x - tx, yy = Y[a].y - ty, yz = Y[a].z - tz;
#pragma unroll
                        for (int i = 0; i < NU; i++) {
                            const float ex = yx - X[i].x, ey = yy - X[i].y, ez = yz - X[i].z;
                            const float d2 = fmaf(ex, ex, fmaf(ey, ey, ez * ez));
                            bm.offer(d2, i, a);
                            if (a == P.iref) brv.offer(d2, i, a);
                            if (i == P.iref) bru.offer(d2, a, i);
                        }
                    }
                };
                if (e.w >= 0) {
                    // one shift, whose centre test the walk has already passed
                    // with the same arithmetic (small molecules: a second
                    // inlined copy of the atom loop is cheap)
                    float tx, ty, tz;
                    shift_of(gh, e.w % 3 - 1, (e.w / 3) % 3 - 1, e.w / 9 - 1, tx, ty, tz);
                    atoms(tx, ty, tz);
                } else {
                    for (int iz = 0; iz < kz; iz++)
                    for (int iy = 0; iy < ky; iy++)
                    for (int ix = 0; ix < kx; ix++) {
                        float tx, ty, tz;
                        shift_of(gh, nth_shift(mxs, ix), nth_shift(mys, iy), nth_shift(mzs, iz), tx, ty, tz);
                        const float dx = cv.x - (cuc.x + tx), dy = cv.y - (cuc.y + ty), dz = cv.z - (cuc.z + tz);
                        if (dx * dx + dy * dy + dz * dz > gh.rpre2) continue;
                        atoms(tx, ty, tz);
                    }
                }
            } else {
                for (int iz = 0; iz < kz; iz++)
                for (int iy = 0; iy < ky; iy++)
                for (int ix = 0; ix < kx; ix++) {
                    float tx, ty, tz;
                    shift_of(gh, nth_shift(mxs, ix), nth_shift(mys, iy), nth_shift(mzs, iz), tx, ty, tz);
                    const float dx = cv.x - (cuc.x + tx), dy = cv.y - (cuc.y + ty), dz = cv.z - (cuc.z + tz);
                    if (dx * dx + dy * dy + dz * dz > gh.rpre2) continue;
#pragma unroll
                    for (int a = 0; a < NU; a++) {
                        const float yx = Y[a].x - tx, yy = Y[a].y - ty, yz = Y[a].z - tz;
#pragma unroll
                        for (int i = 0; i < NU; i++) {
                            const float ex = yx - X[i].x, ey = yy - X[i].y, ez = yz - X[i].z;
                            const float d2 = fmaf(ex, ex, fmaf(ey, ey, ez * ez));
                            bm.offer(d2, i, a);
                            if (a == P.iref) brv.offer(d2, i, a);
                            if (i == P.iref) bru.offer(d2, a, i);
                        }
                    }
                }
            }
        } else {
            for (int iz = 0; iz < kz; iz++)
            for (int iy = 0; iy < ky; iy++)
            for (int ix = 0; ix < kx; ix++) {
                float tx, ty, tz;
                shift_of(gh, nth_shift(mxs, ix), nth_shift(mys, iy), nth_shift(mzs, iz), tx, ty, tz);
                const float dx = cv.x - (cuc.x + tx), dy = cv.y - (cuc.y + ty), dz = cv.z - (cuc.z + tz);
                if (dx * dx + dy * dy + dz * dz > gh.rpre2) continue;
                for (int a = 0; a < P.nv; a++) {
                    const float4 y = yw[a];
                    const float yx = y.x - tx, yy = y.y - ty, yz = y.z - tz;
                    for (int i = 0; i < P.nu; i++) {
                        const float4 s4 = xs[i];
                        const float ex = yx - s4.x, ey = yy - s4.y, ez = yz - s4.z;
                        const float d2 = fmaf(ex, ex, fmaf(ey, ey, ez * ez));
                        bm.offer(d2, i, a);
                        if (a == P.iref) brv.offer(d2, i, a);
                        if (P.self_ && i == P.iref) bru.offer(d2, a, i);
                    }
                }
            }
        }
        if (P.self_) return emit_self(u, v, bm, brv, bru, d0, d1);
        emit(u, v, bm, brv);
        return 0;
    }
};

// Real pass of the many-solute-molecule family.  blockIdx.y is the frame;
// each lane owns one solvent molecule v (self: in cell order).  The lanes walk
// their distinct neighbour cells together (trip count = the wavefront's
// largest cell, four candidates per step with their loads in flight), the
// molecule pairs with a centre within reach under some lattice shift are
// appended to an LDS queue (ballot offsets), and the queue is evaluated 64
// pairs at a time, one pair per lane, so the nu x nv atom loops (over every
// shift that maps the two cells onto each other) run without divergence.
// Self-MDDF evaluates each unordered pair once (u < v) and emits the records
// of both orientations (same distance and argmin pair; reference atoms and tie
// order per orientation).
template <class TU, class TV, int NU>
__global__ void __launch_bounds__(BLOCK, 3) k_eval_mols_real(KP P, Bufs B, const TU* xu, const TV* xv, int gx, int S)
{
    // XCD-aware order: workgroups go round-robin to the 8 XCDs, each with its
    // own L2.  XCD k takes the k-th eighth of the (frame, block) items in
    // frame-major order, so each XCD works through its frames one at a time
    // and its L2 holds the molecules of one frame instead of a slice of
    // every frame of the batch.  gx blocks cover one frame.
    const int items = gx * P.F;
    const int per = (items + 7) >> 3;
    const int item = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if (item >= items) return;   // uniform per block, before any barrier
    const int f = item / gx, bx = item - (item / gx) * gx;
    extern __shared__ unsigned sh[];
    const int gwords = P.glds ? P.nbins * (P.gnu + (P.self_ ? 0 : P.gnv)) : 0;
    hist_clear(sh, 2 * P.nbins + gwords);
    unsigned* shg = P.glds ? sh + 2 * P.nbins : nullptr;
    int4* q = (int4*)(sh + ((2 * P.nbins + gwords + 3) & ~3)) + (threadIdx.x >> 6) * QCAP;
    // self: deferred FP64 entries (two int4 each) after the pair queues
    int4* dq = (int4*)(sh + ((2 * P.nbins + gwords + 3) & ~3)) + (BLOCK / 64) * QCAP + (threadIdx.x >> 6) * 2 * DCAP;
    int dqn = 0;
    const int lane = threadIdx.x & 63;
    const PairCtx<TU, TV, NU> ctx(P, B, f, xu, xv, sh, shg);
    const GeoHot& gh = ctx.gh;
    const float4* srt = B.sorted + (int64_t)f * B.nitems;
    const int* st = B.start + (int64_t)f * (P.cap + 1);
    const int nc[3] = {gh.nc[0], gh.nc[1], gh.nc[2]};
    const int nd[3] = {min(nc[0], 3), min(nc[1], 3), min(nc[2], 3)};
    const bool simple = nc[0] >= 3 && nc[1] >= 3 && nc[2] >= 3;
    constexpr int CU = 8;   // candidates per lane per step
    const int stride = gx * blockDim.x;
    const unsigned long long lt = (1ull << lane) - 1ull;
    // S lanes per solvent molecule (small systems): lane sub of a molecule
    // walks the offsets sub, sub + S, ... of the neighbour walk
    for (int base = bx * blockDim.x + (threadIdx.x & ~63); base < P.Mv * S; base += stride) {
        const int vl = base + lane;
        const int q0 = vl / S, sub = vl - (vl / S) * S;
        const bool act = q0 < P.Mv;
        const int v = act ? (P.self_ ? __float_as_int(srt[q0].w) : q0) : 0;
        const float4 cv = ctx.vcen[v];
        const int vcell = ctx.vcellf[v];
        const int cc[3] = {vcell % nc[0], (vcell / nc[0]) % nc[1], vcell / (nc[0] * nc[1])};
        const int ncells = nd[0] * nd[1] * nd[2];
        // The walk over the neighbour cells produces queue entries until 64
        // are waiting, the wavefront evaluates them, and the walk resumes where
        // it stopped: the pair evaluation has one call site (one inlined copy).
        int qn = 0;
        // Self with three or more cells per dimension: every offset maps to a
        // distinct cell, so each unordered pair of molecules in different
        // cells is met exactly once from the half shell of offsets after
        // (0, 0, 0) (linear index 13 of the 27; z, then y, then x), and pairs
        // inside one cell once with u < v.  Otherwise all offsets with u < v.
        const int o_first = (P.self_ && simple) ? 13 : 0;
        const int nsteps = (ncells - o_first + S - 1) / S;   // walk steps, the same for every lane
        int ks = 0, o = o_first + sub, kpos = 0, kmax = -1;
        int cell = 0, cs = 0, cnt = 0, code = -1, kx = 1, ky = 1, kz = 1;
        int sxs = 0, sys_ = 0, szs = 0;   // shift sets of the current cell (small grids)
        float t1x = 0.f, t1y = 0.f, t1z = 0.f;   // regular grids: own centre minus the cell's shift
        for (;;) {
            while (qn < 64 && ks < nsteps) {
                if (kmax < 0) {
                    // enter neighbour cell o: offsets -1..1, or 0..nc-1 when nc < 3
                    // (a lane whose offsets are used up walks nothing)
                    const bool ov = o < ncells;
                    const int oc = ov ? o : o_first;
                    const int ox = oc % nd[0], oy = (oc / nd[0]) % nd[1], oz = oc / (nd[0] * nd[1]);
                    int m0;
                    const int cx = nb_cell(cc[0], nc[0] >= 3 ? ox - 1 : ox, nc[0], m0);
                    const int cy = nb_cell(cc[1], nc[1] >= 3 ? oy - 1 : oy, nc[1], m0);
                    const int cz = nb_cell(cc[2], nc[2] >= 3 ? oz - 1 : oz, nc[2], m0);
                    cell = (cz * nc[1] + cy) * nc[0] + cx;
                    if (simple) {
                        // three or more cells per dimension: one shift
                        int mx, my, mz;
                        nb_cell(cc[0], ox - 1, nc[0], mx);
                        nb_cell(cc[1], oy - 1, nc[1], my);
                        nb_cell(cc[2], oz - 1, nc[2], mz);
                        code = (mx + 1) + 3 * (my + 1) + 9 * (mz + 1);
                        shift_of(gh, mx, my, mz, t1x, t1y, t1z);
                        // the centre test below is a pre-filter with a margin
                        // (rpre), so its rounding does not matter: the shift is
                        // taken off the lane's own centre once per cell
                        t1x = cv.x - t1x;
                        t1y = cv.y - t1y;
                        t1z = cv.z - t1z;
                    } else {
                        sxs = shifts_onto(cc[0], cx, nc[0]);
                        sys_ = shifts_onto(cc[1], cy, nc[1]);
                        szs = shifts_onto(cc[2], cz, nc[2]);
                        kx = __popc(sxs);
                        ky = __popc(sys_);
                        kz = __popc(szs);
                    }
                    cs = st[cell];
                    cnt = (act && ov) ? st[cell + 1] - cs : 0;
                    kmax = wave_max_i(cnt);
                    kpos = 0;
                }
                if (kpos >= kmax) {
                    ks++;
                    o += S;
                    kmax = -1;
                    continue;
                }
                float4 cu4[CU];
#pragma unroll
                for (int w = 0; w < CU; w++) cu4[w] = srt[min(cs + min(kpos + w, max(cnt - 1, 0)), P.Mu - 1)];
                int w = 0;
#pragma unroll
                for (int ww = 0; ww < CU; ww++) {
                    if (w != ww || kpos + ww >= kmax || qn >= 64) break;
                    const int u = __float_as_int(cu4[ww].w);
                    bool pass = kpos + ww < cnt && (P.self_ ? ((simple && o > 13) || u < v) : true);
                    if (simple) {
                        const float dx = t1x - cu4[ww].x, dy = t1y - cu4[ww].y, dz = t1z - cu4[ww].z;
                        pass = pass && dx * dx + dy * dy + dz * dz <= gh.rpre2;
                    } else if (pass) {
                        bool nearby = false;
                        for (int iz = 0; iz < kz; iz++)
                        for (int iy = 0; iy < ky; iy++)
                        for (int ix = 0; ix < kx; ix++) {
                            float tx, ty, tz;
                            shift_of(gh, nth_shift(sxs, ix), nth_shift(sys_, iy), nth_shift(szs, iz), tx, ty, tz);
                            const float dx = cv.x - (cu4[ww].x + tx), dy = cv.y - (cu4[ww].y + ty),
                                        dz = cv.z - (cu4[ww].z + tz);
                            nearby |= dx * dx + dy * dy + dz * dz <= gh.rpre2;
                        }
                        pass = nearby;
                    }
                    const unsigned long long m = __ballot(pass);
                    if (pass) q[qn + __popcll(m & lt)] = make_int4(u, v, cell, code);
                    qn += __popcll(m);
                    w = ww + 1;
                }
                kpos += w;
            }
            if (qn == 0) break;
            const int ne = min(qn, 64);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            const bool has = lane < ne;
            const int4 e = q[has ? qn - ne + lane : 0];
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            qn -= ne;
            int4 d0 = make_int4(0, 0, 0, 0), d1 = d0;
            int dm = 0;
            if (has) dm = ctx.eval_pair(e, d0, d1);
            if (P.self_) {
                // parts FP32 could not decide wait in the deferred queue and
                // are resolved 64 at a time, so the FP64 work runs on full
                // wavefronts
                const unsigned long long m = __ballot(dm != 0);
                if (dm != 0) {
                    const int k = dqn + __popcll(m & lt);
                    dq[2 * k] = d0;
                    dq[2 * k + 1] = make_int4(d1.x, d1.y, dm, 0);
                }
                dqn += __popcll(m);
                if (dqn >= 64) {
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    const int k = dqn - 64 + lane;
                    const int4 x0 = dq[2 * k], x1 = dq[2 * k + 1];
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    dqn -= 64;
                    ctx.self_deferred(x0, x1, x1.z);
                }
            }
        }
    }
    if (dqn > 0) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        if (lane < dqn) {
            const int4 x0 = dq[2 * lane], x1 = dq[2 * lane + 1];
            ctx.self_deferred(x0, x1, x1.z);
        }
    }
    hist_flush(sh, P.nbins, B.cnt_md, B.cnt_rdf);
    if (shg) groups_flush(P, shg, B.cnt_gu, B.cnt_gv);
}

// ---------------------------------------------------------------------------
// bulk lists and random placement
// ---------------------------------------------------------------------------
// bulk flags: bit 0, in the bulk; bit 1 (tiles family), without a position
constexpr unsigned char BULK_VOID = 2;

__device__ __forceinline__ void b_bulk_init(KP P, Bufs B, int bx_, int nbx_, int by_, int nby_)
{
    int64_t total = (int64_t)P.F * P.kb * P.Mv;
    for (int64_t it = bx_ * (int64_t)blockDim.x + threadIdx.x; it < total; it += (int64_t)nbx_ * blockDim.x) {
        int64_t fk = it / P.Mv;
        int v = (int)(it - fk * P.Mv);
        unsigned char fl = P.usecutoff ? 0 : 1;
        if (P.self_ && B.uk[fk] == v) fl = 0;   // the bulk pool excludes isolute, src/mddf.jl:410
        B.bflag[it] = fl;
    }
}

__global__ void k_bulk_init(KP P, Bufs B)
{
    b_bulk_init(P, B, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// Slots listed per (frame, pass) of the molecule-pair family.  The counts take the
// place of drawn_idx, which the real pass was the last to read.
__device__ __forceinline__ int* slot_counts(const Bufs& B) { return B.drawn_idx; }

// ordered compaction of the bulk flags, one block per (frame, list)
__device__ __forceinline__ void b_bulk_compact(KP P, Bufs B, int bx_, int nbx_, int by_, int nby_, bool mols = false)
{
    if (mols)
        for (int k = bx_ * blockDim.x + threadIdx.x; k < P.F * P.K; k += nbx_ * blockDim.x) slot_counts(B)[k] = 0;
    __shared__ int wsum[16];
    __shared__ int carry;
    int64_t fk = bx_;
    const unsigned char* fl = B.bflag + fk * P.Mv;
    int* out = B.blist + fk * P.Mv;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    // four consecutive flags per thread, the counts scanned over the
    // wavefront (DPP) and across the block's wavefronts
    for (int base = 0; base < P.Mv; base += 4 * blockDim.x) {
        const int v0 = base + 4 * threadIdx.x;
        int fl4[4];
#pragma unroll
        for (int u = 0; u < 4; u++) fl4[u] = v0 + u < P.Mv ? fl[v0 + u] & 1 : 0;
        const int cnt = fl4[0] + fl4[1] + fl4[2] + fl4[3];
        const int incl = wave_incl_scan(cnt);
        if (lane == 63) wsum[wid] = incl;
        __syncthreads();
        int woff = 0, tot = 0;
        for (int w = 0; w < nw; w++) { if (w < wid) woff += wsum[w]; tot += wsum[w]; }
        int o = carry + woff + incl - cnt;
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (fl4[u]) out[o++] = v0 + u;
        __syncthreads();
        if (threadIdx.x == 0) carry += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) B.nbulk[fk] = carry;
}

__global__ void __launch_bounds__(1024) k_bulk_compact(KP P, Bufs B, int mols)
{
    b_bulk_compact(P, B, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y, mols != 0);
}

// The atoms of one source molecule (xyz interleaved) and the placed atoms
// (FP64 for the exact resolve, FP32 for the evaluation), through global
// pointers (also where the pointers were read from a job table).
template <class TV>
struct MolSrc {
    gptr<const TV> p;
    __device__ MolSrc(const TV* q) : p((gptr<const TV>)q) {}
    __device__ double operator()(int a, int k) const { return (double)p[3 * a + k]; }
};

// the same of three atoms, read once (with a constant count random_move's loops
// unroll, and the wrapped positions that it forms twice are formed once)
template <class TV>
struct MolSrc3 {
    TV x[9];
    __device__ MolSrc3(const TV* q)
    {
        const gptr<const TV> p = (gptr<const TV>)q;
#pragma unroll
        for (int k = 0; k < 9; k++) x[k] = p[k];
    }
    __device__ double operator()(int a, int k) const { return (double)(a == 0 ? x[k] : (a == 1 ? x[3 + k] : x[6 + k])); }
};

struct MolDst {
    gptr<double> p;
    float4* w;   // (k_eval_mols_rand reads these in the same thread)
    __device__ MolDst(double* q, float4* v) : p((gptr<double>)q), w(v) {}
    __device__ void operator()(int a, double x, double y, double z) const
    {
        p[3 * a] = x; p[3 * a + 1] = y; p[3 * a + 2] = z;
        w[a] = mk4((float)x, (float)y, (float)z, 0.f);
    }
};

// the same with fixed-point positions for the evaluation
struct MolDstFix {
    gptr<double> p;
    gptr<f4v> w;
    const Geo& g;
    bool keep;   // the FP64 positions too
    __device__ MolDstFix(double* q, float4* v, const Geo& geo, bool k) : p((gptr<double>)q), w((gptr<f4v>)v), g(geo), keep(k) {}
    __device__ void operator()(int a, double x, double y, double z) const
    {
        if (keep) { p[3 * a] = x; p[3 * a + 1] = y; p[3 * a + 2] = z; }
        const float4 u = fix_point(g, x, y, z, 0.f);
        w[a] = f4v{u.x, u.y, u.z, 0.f};
    }
    // the first atom's fourth component
    __device__ void set_w0(float x) const { ((gptr<float>)w)[3] = x; }
};

// the FP64 positions alone
struct MolDst64 {
    gptr<double> p;
    __device__ MolDst64(double* q) : p((gptr<double>)q) {}
    __device__ void operator()(int a, double x, double y, double z) const { p[3 * a] = x; p[3 * a + 1] = y; p[3 * a + 2] = z; }
};

// Whether placed slot v (centre cv) can have an atom pair with the drawn
// solute molecule (centre cu) within the cutoff under some lattice shift: the
// centre pre-check of the random passes of the molecule-pair family.  In a
// diagonal cell the nearest image decides (rounding: rpre2's margin of 1e-2 A).
__device__ __forceinline__ bool mol_pair_near(const Geo& g, float4 cv, float4 cu)
{
    const float dx = cv.x - cu.x, dy = cv.y - cu.y, dz = cv.z - cu.z;
    if (g.ortho) {
        float ox, oy, oz;
        minimage32(g, dx, dy, dz, ox, oy, oz);
        return !(ox * ox + oy * oy + oz * oz > g.rpre2);
    }
    bool any = false;
    for (int mz = -1; mz <= 1; mz++)
    for (int my = -1; my <= 1; my++)
    for (int mx = -1; mx <= 1; mx++) {
        const float fx = (float)mx, fy = (float)my, fz = (float)mz;
        const float ex = dx - (g.H32[0] * fx + g.H32[3] * fy + g.H32[6] * fz);
        const float ey = dy - (g.H32[1] * fx + g.H32[4] * fy + g.H32[7] * fz);
        const float ez = dz - (g.H32[2] * fx + g.H32[5] * fy + g.H32[8] * fz);
        any |= !(ex * ex + ey * ey + ez * ez > g.rpre2);
    }
    return any;
}

// The slots of the random passes that can be within the cutoff of their drawn
// solute molecule (all of them when the placements are kept for verification),
// listed per (frame, pass).  A few per cent are; placed and evaluated where
// they lie, one or two lanes of a wavefront would work at a time.  16,667 waters
// about 181 osmolytes, 20 frames of 10 passes: placement 125 and evaluation
// 229 us so, 25 us for the list (random numbers and the test) and 68 us for
// both now; with an atomic per wavefront the list alone took 217 us.
constexpr int NEAR_SLOTS = 4;   // slots per thread: one atomic a block (each takes about 10 ns of its line's time)
__global__ void __launch_bounds__(BLOCK) k_mols_near(KP P, Bufs B)
{
    // grid: x over the slots, y over the (frame, pass) pairs
    __shared__ float4 list[NEAR_SLOTS * BLOCK];
    __shared__ int n, base;
    const int v0 = blockIdx.x * NEAR_SLOTS * BLOCK, lane = threadIdx.x & 63;
    for (int fk = blockIdx.y; fk < P.F * P.K; fk += gridDim.y) {
        const int f = fk / P.K;
        const int k = fk - f * P.K;
        const Geo& g = B.geo[f];
        const int u = B.uk[fk];
        const float4 cu = B.ucen[(int64_t)f * P.Mu + u];
        const double* H = g.cell.H;
        if (threadIdx.x == 0) n = 0;
        __syncthreads();
        for (int v = v0 + threadIdx.x; v < v0 + NEAR_SLOTS * BLOCK; v += BLOCK) {
            const cm::u32x4 r = cm::philox4x32_10({(uint32_t)v, (uint32_t)k, g.frame, cm::TAG_SLOT}, P.key0, P.key1);
            const double uc[3] = {cm::u01(r.y), cm::u01(r.z), cm::u01(r.w)};
            // the new centre H*uc (inside the cell)
            const double c0 = H[0] * uc[0] + H[3] * uc[1] + H[6] * uc[2];
            const double c1 = H[1] * uc[0] + H[4] * uc[1] + H[7] * uc[2];
            const double c2 = H[2] * uc[0] + H[5] * uc[1] + H[8] * uc[2];
            const float4 cv = mk4((float)c0, (float)c1, (float)c2, __int_as_float(v));
            const bool take = v < P.Mv && (P.place_all || (!(P.self_ && u == v) && mol_pair_near(g, cv, cu)));
            const unsigned long long m = __ballot(take);
            if (!m) continue;
            int o = 0;
            if (lane == 0) o = atomicAdd(&n, __popcll(m));
            o = __builtin_amdgcn_readfirstlane(o);
            if (take) list[o + __popcll(m & ((1ull << lane) - 1ull))] = cv;
        }
        __syncthreads();
        if (threadIdx.x == 0) base = n ? atomicAdd(&slot_counts(B)[fk], n) : 0;
        __syncthreads();
        for (int e = threadIdx.x; e < n; e += BLOCK) B.vcen_r[(int64_t)fk * P.Mv + base + e] = list[e];
        __syncthreads();
    }
}

// The listed slots, one thread each: placement (randomize_solvent!,
// src/mddf.jl:65-88) and the record of the drawn solute molecule with the
// placed one.  blockIdx.y: (frame, pass) pairs; the wavefronts of the blocks of
// a pair take 64 slots in turn.  A launch has one or two turns: bound by the
// latency of one (FP64 rotation, minima, records) and the flush of the blocks'
// few counts.
template <class TU, class TV>
__global__ void __launch_bounds__(BLOCK) k_eval_mols_rand(KP P, Bufs B, const TU* xu, const TV* xv)
{
    extern __shared__ unsigned sh[];
    const int gwords = P.glds ? P.nbins * (P.gnu + (P.self_ ? 0 : P.gnv)) : 0;
    hist_clear(sh, 2 * P.nbins + gwords);
    unsigned* shg = P.glds ? sh + 2 * P.nbins : nullptr;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int fk = blockIdx.y; fk < P.F * P.K; fk += gridDim.y) {
        const int f = fk / P.K;
        const int k = fk - f * P.K;
        const Geo& g = B.geo[f];
        const int u = B.uk[fk], count = slot_counts(B)[fk];
        const int64_t lk = (int64_t)f * P.kb + (P.kb == 1 ? 0 : k);
        const int nb = B.nbulk[lk];
        const float4 cu = B.ucen[(int64_t)f * P.Mu + u];
        const float4* xs = B.solw + (int64_t)f * P.Nu + (int64_t)u * P.nu;
        for (int n = (wid * gridDim.x + blockIdx.x) * 64 + lane; n < count; n += nw * gridDim.x * 64) {
            const float4 cv = B.vcen_r[(int64_t)fk * P.Mv + n];
            const int v = __float_as_int(cv.w);
            const cm::u32x4 r = cm::philox4x32_10({(uint32_t)v, (uint32_t)k, g.frame, cm::TAG_SLOT}, P.key0, P.key1);
            const cm::u32x4 r2 = cm::philox4x32_10({(uint32_t)v, (uint32_t)k, g.frame, cm::TAG_SLOT + 1u}, P.key0, P.key1);
            const double uc[3] = {cm::u01(r.y), cm::u01(r.z), cm::u01(r.w)};
            const double ua[3] = {cm::u01(r2.x), cm::u01(r2.y), cm::u01(r2.z)};
            const int64_t jmol = nb > 0 ? (int64_t)B.blist[lk * P.Mv + cm::draw_index(r.x, nb)] : cm::draw_index(r.x, P.Mv);
            MolSrc<TV> src(xv + (int64_t)f * P.Nv * 3 + jmol * P.nv * 3);
            const int64_t jbase = (int64_t)v * P.nv;
            MolDst dst(B.P + (fk * (int64_t)P.Nv + jbase) * 3, B.vw_r + fk * (int64_t)P.Nv + jbase);
            cm::random_move(src, dst, P.nv, P.iref, g.cell, uc, ua);
            if ((P.self_ && u == v) || (P.place_all && !mol_pair_near(g, cv, cu))) continue;
            const float4* yw = B.vw_r + fk * (int64_t)P.Nv + jbase;
            Best bm, br;
            bm.init(); br.init();
            // the lattice shifts in reach, then a shift of its own per lane and turn
            unsigned near = 0;
            for (int q = 0; q < 27; q++) {
                const float fx = (float)(q % 3 - 1), fy = (float)(q / 3 % 3 - 1), fz = (float)(q / 9 - 1);
                const float dx = cv.x - (cu.x + (g.H32[0] * fx + g.H32[3] * fy + g.H32[6] * fz));
                const float dy = cv.y - (cu.y + (g.H32[1] * fx + g.H32[4] * fy + g.H32[7] * fz));
                const float dz = cv.z - (cu.z + (g.H32[2] * fx + g.H32[5] * fy + g.H32[8] * fz));
                near |= dx * dx + dy * dy + dz * dz > g.rpre2 ? 0u : 1u << q;
            }
            for (; near; near &= near - 1) {
                const int q = __builtin_ctz(near);
                const float fx = (float)(q % 3 - 1), fy = (float)(q / 3 % 3 - 1), fz = (float)(q / 9 - 1);
                pairs_mol(P, xs, yw, g.H32[0] * fx + g.H32[3] * fy + g.H32[6] * fz, g.H32[1] * fx + g.H32[4] * fy + g.H32[7] * fz,
                          g.H32[2] * fx + g.H32[5] * fy + g.H32[8] * fz, bm, br);
            }
            const TU* xuf = xu + (int64_t)f * P.Nu * 3;
            auto ysrc = [&](int a, double& y0, double& y1, double& y2) {
                const double* pp = B.P + (fk * (int64_t)P.Nv + jbase + a) * 3; y0 = pp[0]; y1 = pp[1]; y2 = pp[2];
            };
            Rec rec = resolve_mols(P, g, xuf, u, v, ysrc, bm, br, &B.stats[0]);
            hist_record_mols(P, sh, shg, B.cnt_gu_r, B.cnt_gv_r, rec);
        }
    }
    hist_flush(sh, P.nbins, B.cnt_md_r, B.cnt_rdf_r);
    if (shg) groups_flush(P, shg, B.cnt_gu_r, B.cnt_gv_r);
}

// ---------------------------------------------------------------------------
// tiles family: one solute molecule, solvent molecules of up to 64 atoms
// ---------------------------------------------------------------------------
constexpr int RB_PIECES = 8;        // read-back pieces of cm_job_finish
constexpr int CBCAP = 1024;         // chunk-table entries kept in LDS
// The last DYN_PCT per cent of an evaluation launch's chunks are handed out
// on request, in launches of at least DYN_MIN chunks per workgroup, in about
// DYN_GRABS requests per workgroup (consecutive chunks per request).  On the
// 200-frame globule job and 64 uneven systems (random-pass launch time):
// 35% in requests of one chunk -9%, of two (8 requests) -17%, of four -12%;
// 25% -11%, 45% (two per request) -17%, 55% and more in single chunks slower
// than a fixed stride alone.
constexpr int DYN_PCT = 35;
constexpr int DYN_MIN = 2;
constexpr int DYN_GRABS = 8;

__device__ __forceinline__ int wrap_index(int i, int n, int& m)
{
    int q = i >= 0 ? i / n : -((-i + n - 1) / n);
    m = q;
    return i - q * n;
}

// Sort keys: the position of a fine cell (or half-cell) on the Hilbert curve of
// its grid, so that consecutive molecules stay compact in space (a run of 64
// near molecules of ten merged passes: boxes of 8.6 A a side and 166 staged
// solute atoms, against 11.0 A and 288 along the Morton curve).  HILBERT[state][octant]: the
// octant's place among the eight of its parent cube (bits 0..2) and the state
// of its own eight (bits 3..7), the 24 orientations of the curve of Skilling,
// "Programming the Hilbert curve" (AIP Conf. Proc. 707, 2004).
__device__ const __align__(16) unsigned char HILBERT[24 * 8] = {
    0x08, 0x3f, 0x23, 0x2c, 0x19, 0x36, 0x02, 0x05,
    0x10, 0xab, 0x41, 0x0a, 0x57, 0x1c, 0x5e, 0x0d,
    0x00, 0x29, 0x77, 0x6e, 0x63, 0x12, 0x44, 0x15,
    0x28, 0x8b, 0x6f, 0x0c, 0x01, 0x1a, 0x76, 0x1d,
    0x86, 0x47, 0x25, 0x4c, 0xb1, 0x58, 0x22, 0x03,
    0x40, 0x11, 0x4b, 0x2a, 0x5f, 0x56, 0x04, 0x2d,
    0x7c, 0x27, 0x3b, 0xa0, 0x35, 0x06, 0x32, 0x71,
    0xbc, 0x87, 0x3d, 0x46, 0x33, 0xb0, 0x3a, 0x59,
    0x18, 0x37, 0x09, 0x3e, 0x83, 0x14, 0x42, 0x45,
    0xae, 0xb9, 0x4d, 0x4a, 0x0f, 0x38, 0x24, 0x2b,
    0x94, 0x55, 0x5b, 0x52, 0x4f, 0x2e, 0x98, 0x69,
    0xb4, 0x53, 0x5d, 0x5a, 0xaf, 0xb8, 0x0e, 0x39,
    0x8e, 0x79, 0x1f, 0x30, 0x65, 0x62, 0x84, 0x13,
    0x9c, 0x6d, 0x67, 0x16, 0x73, 0x6a, 0x90, 0x51,
    0xa4, 0x6b, 0x8f, 0x78, 0x75, 0x72, 0x1e, 0x31,
    0x7a, 0x61, 0xbb, 0x80, 0x7d, 0x96, 0x34, 0xb7,
    0x26, 0x07, 0xa1, 0x70, 0x85, 0x64, 0x82, 0x43,
    0x66, 0x8d, 0x17, 0xac, 0x91, 0x8a, 0x50, 0x1b,
    0x92, 0x95, 0xb3, 0x54, 0x89, 0x7e, 0xa8, 0xbf,
    0x9a, 0x9d, 0xa9, 0xbe, 0xa3, 0x6c, 0x88, 0x7f,
    0xa2, 0x9b, 0x81, 0x60, 0xa5, 0x74, 0xb6, 0x97,
    0x4e, 0xad, 0x99, 0xaa, 0x2f, 0x8c, 0x68, 0x0b,
    0xb2, 0x93, 0xb5, 0x5c, 0x21, 0x48, 0xa6, 0x9f,
    0xba, 0x49, 0xbd, 0x9e, 0x7b, 0x20, 0x3c, 0xa7,
};

// the table in LDS (48 words), for a kernel whose lanes walk it
__device__ __forceinline__ void hilbert_load(unsigned* tab)
{
    if (threadIdx.x < 48) tab[threadIdx.x] = ((const unsigned*)HILBERT)[threadIdx.x];
    __syncthreads();
}

// key of the cell (c0, c1, c2), each below 2^bits; tab: hilbert_load's
__device__ __forceinline__ int hilbert_key(const unsigned* tab, int bits, int c0, int c1, int c2)
{
    const unsigned char* t = (const unsigned char*)tab;
    int key = 0, state = 0;
    for (int b = bits - 1; b >= 0; b--) {
        const int o = ((c0 >> b) & 1) | (((c1 >> b) & 1) << 1) | (((c2 >> b) & 1) << 2);
        const int e = t[state * 8 + o];
        key = (key << 3) | (e & 7);
        state = e >> 3;
    }
    return key;
}

// Fine-grid index ranges covering the box [lo - r, hi + r] (fractional
// coordinates of its 8 corners, with a small outward margin).
__device__ __forceinline__ void cell_range(const Geo& g, float lx, float ly, float lz, float hx, float hy, float hz,
                                           float r, int ilo[3], int ihi[3])
{
    const double* Hi = g.cell.Hi;
    double fmn[3] = {INFINITY, INFINITY, INFINITY}, fmx[3] = {-INFINITY, -INFINITY, -INFINITY};
    if (g.ortho) {
        // diagonal cell: the corners' fractional coordinates are the two
        // products per dimension (the off-diagonal terms are exact zeros, so
        // the values equal the general form's)
        const double lo3[3] = {(double)lx - r, (double)ly - r, (double)lz - r};
        const double hi3[3] = {(double)hx + r, (double)hy + r, (double)hz + r};
        for (int k = 0; k < 3; k++) {
            const double a = Hi[4 * k] * lo3[k], b = Hi[4 * k] * hi3[k];
            ilo[k] = (int)floor(fmin(a, b) * g.nc[k] - 1e-6);
            ihi[k] = (int)floor(fmax(a, b) * g.nc[k] + 1e-6);
        }
        return;
    }
    for (int c = 0; c < 8; c++) {
        double x = (c & 1) ? (double)hx + r : (double)lx - r;
        double y = (c & 2) ? (double)hy + r : (double)ly - r;
        double z = (c & 4) ? (double)hz + r : (double)lz - r;
        double f[3] = {Hi[0] * x + Hi[3] * y + Hi[6] * z, Hi[1] * x + Hi[4] * y + Hi[7] * z,
                       Hi[2] * x + Hi[5] * y + Hi[8] * z};
        for (int k = 0; k < 3; k++) { fmn[k] = fmin(fmn[k], f[k]); fmx[k] = fmax(fmx[k], f[k]); }
    }
    for (int k = 0; k < 3; k++) {
        ilo[k] = (int)floor(fmn[k] * g.nc[k] - 1e-6);
        ihi[k] = (int)floor(fmx[k] * g.nc[k] + 1e-6);
    }
}


// The same in FP32 for a box of half sides ex, ey, ez (radius included) about a
// fixed-point centre, widened by more than its rounding (a few 1e-4 cells at
// the largest grids), and kept to the images that an atom within a cell of the
// home cell can reach
template <class GEO>
__device__ __forceinline__ void cell_range32(const GEO& g, int cx, int cy, int cz, float ex, float ey, float ez, int ilo[3],
                                             int ihi[3])
{
    const int c[3] = {cx, cy, cz};
    const float unit = ldexpf(1.0f, -g.fix);
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float m = (float)c[k] * unit;
        const float e = fabsf(g.Hi32[k]) * ex + fabsf(g.Hi32[3 + k]) * ey + fabsf(g.Hi32[6 + k]) * ez;
        const float n = (float)g.nc[k];
        ilo[k] = max((int)floorf((m - e) * n - 2e-3f), -8 * g.nc[k]);
        ihi[k] = min((int)floorf((m + e) * n + 2e-3f), 9 * g.nc[k]);
    }
}

// Lanes an atom in k_near_mark.  Few atoms: eight, each with an eighth of the
// serial walk over the atom's cells (30 atoms: 25 -> 11 us).  From a block's worth
// on, one: the cell ranges that every lane forms are extra (1,000 atoms: 36 us,
// 45 with eight; 5,000: 47 and 65).
__host__ __device__ __forceinline__ int near_lanes(int nu) { return nu < 256 ? 8 : 1; }
constexpr int NEAR_WORDS = 8192;   // LDS bitmap words (frames of up to 262,144 cells; larger: direct stores)

// cells near the solute: every cell within rnear of a solute atom (index
// box).  A block takes 256 consecutive atoms of one frame (neighbours along
// the chain, whose cell ranges overlap): the marks go into a bitmap of the
// frame's cells in LDS first, and the block writes each marked cell once.
__device__ __forceinline__ void b_near_mark(KP P, Bufs B, int bx_, int nbx_, int by_, int nby_)
{
    __shared__ unsigned bits[NEAR_WORDS];
    for (int f = by_; f < P.F; f += nby_) {
        const Geo g = ldc_geo(B.geo + f);
        const int ncell = g.nc[0] * g.nc[1] * g.nc[2];
        const bool lds = ncell <= NEAR_WORDS * 32;
        const int nw = (ncell + 31) >> 5;
        if (lds)
            for (int w = threadIdx.x; w < nw; w += blockDim.x) bits[w] = 0u;
        __syncthreads();
        unsigned char* nr = B.near + (int64_t)f * P.cap;
        // boxes of a diagonal cell: only the cells whose box is within rnear
        // (in the image of index i); otherwise the whole index box
        const float rn2 = g.rnear * g.rnear;
        const float hx = g.H32[0] / g.nc[0], hy = g.H32[4] / g.nc[1], hz = g.H32[8] / g.nc[2];
        auto gap = [](float v, float lo, float hi) { return fmaxf(fmaxf(lo - v, v - hi), 0.f); };
        // cells a..b (0 <= a <= b < nc0) of the row starting at cell rb: a
        // bit range, one LDS atomic per word
        auto mark_run = [&](int rb, int a, int b) {
            const int c0 = rb + a, c1 = rb + b;
            if (lds) {
                for (int w = c0 >> 5; w <= (c1 >> 5); w++) {
                    const int lo = w == (c0 >> 5) ? (c0 & 31) : 0, hi = w == (c1 >> 5) ? (c1 & 31) : 31;
                    const unsigned m = (hi == 31 ? 0xffffffffu : (2u << hi) - 1u) & ~((1u << lo) - 1u);
                    atomicOr(&bits[w], m);
                }
            } else {
                for (int c = c0; c <= c1; c++) nr[c] = 1;
            }
        };
        // a few lanes an atom take its layers of cells in turn
        const int lanes = near_lanes(P.nu);
        for (int64_t e = bx_ * (int64_t)blockDim.x + threadIdx.x; e < (int64_t)P.nu * lanes; e += (int64_t)nbx_ * blockDim.x) {
            const int64_t at = e / lanes;
            const float4 u = B.tmp4[(int64_t)f * P.nu + at];
            if (__float_as_int(u.w) < 0) continue;   // no position
            float4 s;
            fix_cart(g, __float_as_int(u.x), __float_as_int(u.y), __float_as_int(u.z), s.x, s.y, s.z);
            int ilo[3], ihi[3];
            cell_range(g, s.x, s.y, s.z, s.x, s.y, s.z, g.rnear, ilo, ihi);
            for (int iz = ilo[2] + (int)(e % lanes); iz <= ihi[2]; iz += lanes) {
                int mz; int cz = wrap_index(iz, g.nc[2], mz);
                const float dz = g.ortho ? gap(s.z, iz * hz, (iz + 1) * hz) : 0.f;
                for (int iy = ilo[1]; iy <= ihi[1]; iy++) {
                    int my; int cy = wrap_index(iy, g.nc[1], my);
                    const float dy = g.ortho ? gap(s.y, iy * hy, (iy + 1) * hy) : 0.f;
                    const float r2 = rn2 - dz * dz - dy * dy;
                    if (r2 < 0.f) continue;
                    // the x cells of the row within rnear (diagonal cells: their
                    // box gap <= sqrt(r2), widened over FP32 rounding, which
                    // only adds cells), as at most two runs of wrapped cells
                    int x0 = ilo[0], x1 = ihi[0];
                    if (g.ortho) {
                        const float rx = sqrtf(r2) * (1.0f + 1e-6f) + 1e-4f;
                        x0 = max(x0, (int)floorf((s.x - rx) / hx));
                        x1 = min(x1, (int)floorf((s.x + rx) / hx));
                    }
                    if (x0 > x1) continue;
                    const int rb = (cz * g.nc[1] + cy) * g.nc[0];
                    if (x1 - x0 + 1 >= g.nc[0]) {
                        mark_run(rb, 0, g.nc[0] - 1);
                    } else {
                        int m0, m1;
                        const int a = wrap_index(x0, g.nc[0], m0), b = wrap_index(x1, g.nc[0], m1);
                        if (a <= b) {
                            mark_run(rb, a, b);
                        } else {
                            mark_run(rb, a, g.nc[0] - 1);
                            mark_run(rb, 0, b);
                        }
                    }
                }
            }
        }
        __syncthreads();
        if (lds)
            for (int w = threadIdx.x; w < nw; w += blockDim.x) {
                unsigned m = bits[w];
                while (m) {
                    const int bit = __ffs(m) - 1;
                    m &= m - 1u;
                    nr[(w << 5) + bit] = 1;
                }
            }
        __syncthreads();
    }
}

__global__ void k_near_mark(KP P, Bufs B)
{
    b_near_mark(P, B, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// Every near cell: the distance from its centre q to the nearest image of a
// solute atom in the cell itself or one of its six face neighbours, and the
// distance from its lower corner to the nearest image in the eight cells
// around that corner; each encoded as 0xffffffff - bits (0, the cleared
// value, when the cells hold no atom).  Each is the distance to one
// particular atom image, so for any point p min_a |p - a| <= |p - q| + that
// distance: each molecule of the cell gets from them an upper bound on its
// atoms' nearest solute distance (molecule_bound).  Sixteen lanes per cell:
// lane j < 7 scans one cell for the centre, lane 8 + t one for the corner.
__device__ __forceinline__ void b_dfield(KP P, Bufs B, int bx_, int nbx_, int by_, int nby_)
{
    const int64_t total = (int64_t)P.F * P.cap;
    const int j = threadIdx.x & 15;
    const int64_t step = ((int64_t)nbx_ * blockDim.x) >> 4;
    // the sixteen lanes of a group share it (blockDim is a multiple of 16)
    for (int64_t it = (bx_ * (int64_t)blockDim.x + threadIdx.x) >> 4; it < total; it += step) {
        const bool nearc = B.near[it] != 0;
        float best = INFINITY;
        if (nearc && j != 7) {
            const int f = (int)(it / P.cap);
            const int cell = (int)(it - (int64_t)f * P.cap);
            const Geo g = ldc_geo(B.geo + f);
            const int cx = cell % g.nc[0], cy = (cell / g.nc[0]) % g.nc[1], cz = cell / (g.nc[0] * g.nc[1]);
            int ax, ay, az;
            float fx, fy, fz;
            if (j < 7) {
                ax = j == 1 ? 1 : (j == 2 ? -1 : 0);
                ay = j == 3 ? 1 : (j == 4 ? -1 : 0);
                az = j == 5 ? 1 : (j == 6 ? -1 : 0);
                fx = (cx + 0.5f) / g.nc[0]; fy = (cy + 0.5f) / g.nc[1]; fz = (cz + 0.5f) / g.nc[2];
            } else {
                const int t = j - 8;
                ax = -(t & 1); ay = -((t >> 1) & 1); az = -((t >> 2) & 1);
                fx = (float)cx / g.nc[0]; fy = (float)cy / g.nc[1]; fz = (float)cz / g.nc[2];
            }
            int mx, my, mz;
            const int ix = wrap_index(cx + ax, g.nc[0], mx), iy = wrap_index(cy + ay, g.nc[1], my),
                      iz = wrap_index(cz + az, g.nc[2], mz);
            float tx, ty, tz;
            shift_of(g, mx, my, mz, tx, ty, tz);
            // the reference point minus the image shift, against the wrapped atoms
            const float rx = g.H32[0] * fx + g.H32[3] * fy + g.H32[6] * fz - tx;
            const float ry = g.H32[1] * fx + g.H32[4] * fy + g.H32[7] * fz - ty;
            const float rz = g.H32[2] * fx + g.H32[5] * fy + g.H32[8] * fz - tz;
            const int* st = B.start + (int64_t)f * (P.cap + 1);
            const float4* srt = B.sorted + (int64_t)f * B.nitems;
            const int c2 = (iz * g.nc[1] + iy) * g.nc[0] + ix;
            const int k0 = st[c2], k1 = st[c2 + 1];
            int k = k0;
            auto dist = [&](const float4& a) {
                float ex, ey, ez;
                fix_cart(g, __float_as_int(a.x), __float_as_int(a.y), __float_as_int(a.z), ex, ey, ez);
                ex -= rx; ey -= ry; ez -= rz;
                best = fminf(best, ex * ex + ey * ey + ez * ez);
            };
            for (; k + 3 < k1; k += 4) {
                float4 a[4];
#pragma unroll
                for (int u = 0; u < 4; u++) a[u] = srt[k + u];
#pragma unroll
                for (int u = 0; u < 4; u++) dist(a[u]);
            }
            for (; k < k1; k++) dist(srt[k]);
        }
        // minimum over each eight-lane half (centre: lanes 0-6, corner: 8-15)
        best = fminf(best, __shfl_xor(best, 1, 64));
        best = fminf(best, __shfl_xor(best, 2, 64));
        best = fminf(best, __shfl_xor(best, 4, 64));
        if (nearc && (j & 7) == 0 && best < INFINITY)
            B.dfield[(j ? total : 0) + it] = 0xffffffffu - __float_as_uint(sqrtf(best));
    }
}

__global__ void k_dfield(KP P, Bufs B)
{
    b_dfield(P, B, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// Upper bound (FP32, rounded outward by a wide margin) on the distance from
// any atom of a molecule whose centre has fractional coordinates fr (in the
// near cell `cell`) to its nearest solute atom: the smallest, over the cell's
// centre and its eight corners, of the reference point's atom distance plus
// the distance from the centre to the point, plus the molecule radius; +inf
// when none has a distance.  FP32 throughout: every rounding is far below the
// 1e-5 relative + 0.01 A margin.
struct BoundLoads {
    unsigned e[9];   // the centre's entry, then the corners (a + 2 b + 4 c)
};

// the entries, read by the callers before their stores (which may alias them
// as far as the compiler knows, and would hold the loads back)
__device__ __forceinline__ BoundLoads bound_loads(const KP& P, const Bufs& B, const Geo& g, int f, int cell, int c0,
                                                  int c1, int c2)
{
    // cell = (c2 nc1 + c1) nc0 + c0
    BoundLoads L;
    const gptr<const unsigned> d = (gptr<const unsigned>)(B.dfield + (int64_t)f * P.cap);
    const gptr<const unsigned> dc = d + (int64_t)P.F * P.cap;
    L.e[0] = d[cell];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        int i0 = c0 + (t & 1), i1 = c1 + ((t >> 1) & 1), i2 = c2 + ((t >> 2) & 1);
        if (i0 == g.nc[0]) i0 = 0;
        if (i1 == g.nc[1]) i1 = 0;
        if (i2 == g.nc[2]) i2 = 0;
        L.e[1 + t] = dc[(i2 * g.nc[1] + i1) * g.nc[0] + i0];
    }
    return L;
}

__device__ __forceinline__ float molecule_bound(const Geo& g, const BoundLoads& L, int c0, int c1, int c2,
                                                const double fr[3])
{
    const float* H = g.H32;
    // (hardware reciprocals, 1 ulp: a relative 2^-23 in the offsets below is
    // far inside the bound's margin)
    const float i0 = __builtin_amdgcn_rcpf((float)g.nc[0]), i1 = __builtin_amdgcn_rcpf((float)g.nc[1]),
                i2 = __builtin_amdgcn_rcpf((float)g.nc[2]);
    // centre -> cell centre, and the half-cell steps along the three cell
    // vectors: centre -> corner (a, b, c) = e + (2a - 1) h0 + (2b - 1) h1 + (2c - 1) h2
    const float d0 = (float)fr[0] - (c0 + 0.5f) * i0, d1 = (float)fr[1] - (c1 + 0.5f) * i1,
                d2 = (float)fr[2] - (c2 + 0.5f) * i2;
    const float ex = H[0] * d0 + H[3] * d1 + H[6] * d2;
    const float ey = H[1] * d0 + H[4] * d1 + H[7] * d2;
    const float ez = H[2] * d0 + H[5] * d1 + H[8] * d2;
    const float h0x = 0.5f * i0 * H[0], h0y = 0.5f * i0 * H[1], h0z = 0.5f * i0 * H[2];
    const float h1x = 0.5f * i1 * H[3], h1y = 0.5f * i1 * H[4], h1z = 0.5f * i1 * H[5];
    const float h2x = 0.5f * i2 * H[6], h2y = 0.5f * i2 * H[7], h2z = 0.5f * i2 * H[8];
    float best = INFINITY;
    if (L.e[0] != 0u) best = __uint_as_float(0xffffffffu - L.e[0]) + sqrtf(ex * ex + ey * ey + ez * ez);
#pragma unroll
    for (int t = 0; t < 8; t++) {
        if (L.e[1 + t] == 0u) continue;
        const float sa = (t & 1) ? 1.0f : -1.0f, sb = (t & 2) ? 1.0f : -1.0f, sc = (t & 4) ? 1.0f : -1.0f;
        const float qx = ex - sa * h0x - sb * h1x - sc * h2x;
        const float qy = ey - sa * h0y - sb * h1y - sc * h2y;
        const float qz = ez - sa * h0z - sb * h1z - sc * h2z;
        best = fminf(best, __uint_as_float(0xffffffffu - L.e[1 + t]) + sqrtf(qx * qx + qy * qy + qz * qz));
    }
    if (!(best < INFINITY)) return INFINITY;
    return (best + __uint_as_float(g.rv_bits)) * (1.0f + 1e-5f) + 1e-2f;
}

// real pass: centre of every solvent molecule (made whole around its first
// atom) wrapped into the cell; near molecules get the Hilbert key of the cell
template <class T>
__device__ __forceinline__ void b_prep_solvent_tiles(KP P, Bufs B, const T* xv, const unsigned* tab, int bx_, int nbx_, int by_, int nby_)
{
    int64_t total = (int64_t)P.F * P.Mv;
    for (int64_t it = bx_ * (int64_t)blockDim.x + threadIdx.x; it < total; it += (int64_t)nbx_ * blockDim.x) {
        int f = (int)(it / P.Mv);
        int v = (int)(it - (int64_t)f * P.Mv);
        const Geo g = ldc_geo(B.geo + f);
        double c[3];
        mol_centre(g, xv + (int64_t)f * P.Nv * 3, (int64_t)v * P.nv, P.nv, c);
        double fr[3], n[3];
        wrap_point(g, c[0], c[1], c[2], fr, n);
        int64_t kb = (int64_t)f * P.NP * P.Mv + v;
        if (undefined3(fr)) {
            // no centre (an atom's coordinate is no number): the molecule and
            // what is placed from it (b_place_keys) are within no cutoff
            B.mkey[kb] = -1;
            atomicOr(&B.geo[f].voids, 1u);
            if (P.K > 0) B.bflag[(int64_t)f * P.kb * P.Mv + v] |= BULK_VOID;
            continue;
        }
        int cell, c0, c1, c2;
        cell_of_frac(g, fr[0], fr[1], fr[2], cell, c0, c1, c2);
        if (!B.near[(int64_t)f * P.cap + cell]) { B.mkey[kb] = -1; continue; }
        const int key = hilbert_key(tab, g.kbits, c0, c1, c2);
        B.mkey[kb] = key;
        B.mrank[kb] = atomicAdd(&B.mcnt[key_row(P, f, 0) + key], 1);
    }
}

template <class T>
__global__ void k_prep_solvent_tiles(KP P, Bufs B, const T* xv)
{
    __shared__ unsigned tab[48];
    hilbert_load(tab);
    b_prep_solvent_tiles<T>(P, B, xv, tab, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// real pass: atoms of the near molecules in sorted order, in fixed point (fix_point),
// by the periodic image of the molecule's centre
template <class T>
__device__ __forceinline__ void b_fill_real(KP P, Bufs B, const T* xv, int bx_, int nbx_, int by_, int nby_)
{
    int64_t total = (int64_t)P.F * P.Mv;
    for (int64_t it = bx_ * (int64_t)blockDim.x + threadIdx.x; it < total; it += (int64_t)nbx_ * blockDim.x) {
        int f = (int)(it / P.Mv);
        int pos = (int)(it - (int64_t)f * P.Mv);
        const int64_t fp = (int64_t)f * P.NP;
        if (pos >= B.nnear[(int64_t)f * (1 + P.NG)]) continue;
        const int v = B.msorted[fp * P.Mv + pos];
        const Geo g = ldc_geo(B.geo + f);
        const T* x = xv + (int64_t)f * P.Nv * 3;
        int64_t a0 = (int64_t)v * P.nv;
        double c[3];
        mol_centre(g, x, a0, P.nv, c);
        double fr[3], n[3];
        wrap_point(g, c[0], c[1], c[2], fr, n);
        const double* H = g.cell.H;
        double tx = H[0] * n[0] + H[3] * n[1] + H[6] * n[2];
        double ty = H[1] * n[0] + H[4] * n[1] + H[7] * n[2];
        double tz = H[2] * n[0] + H[5] * n[1] + H[8] * n[2];
        double x0, y0, z0;
        load3(x, a0, x0, y0, z0);
        // the first atom's w carries the molecule's nearest-solute bound
        int cell, c0, c1, c2;
        cell_of_frac(g, fr[0], fr[1], fr[2], cell, c0, c1, c2);
        const float ub = molecule_bound(g, bound_loads(P, B, g, f, cell, c0, c1, c2), c0, c1, c2, fr);
        float4* dst = B.vw + (int64_t)f * P.Nv + (int64_t)pos * P.nv;
        for (int a = 0; a < P.nv; a++) {
            double xa, ya, za, ox, oy, oz;
            load3(x, a0 + a, xa, ya, za);
            cm::minimage(g.cell, xa - x0, ya - y0, za - z0, &ox, &oy, &oz);
            dst[a] = fix_point(g, x0 + ox - tx, y0 + oy - ty, z0 + oz - tz, a == 0 ? ub : 0.f);
        }
    }
}

template <class T>
__global__ void k_fill_real(KP P, Bufs B, const T* xv)
{
    b_fill_real<T>(P, B, xv, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// Keys per part of a row scan: a row is scanned by one block per part, at
// most SCAN_PARTS of them, each part a multiple of 4096 keys (one step of the block).
constexpr int SCAN_PARTS = 512;
__host__ __device__ __forceinline__ int scan_part(int n)
{
    const int p = (n + SCAN_PARTS - 1) / SCAN_PARTS;
    return p <= 8192 ? 8192 : (p + 4095) / 4096 * 4096;
}
__host__ __device__ __forceinline__ int scan_parts(int n) { return (n + scan_part(n) - 1) / scan_part(n); }

// first part of row r of frame f in msum
__device__ __forceinline__ int64_t part_row(const KP& P, int f, int r)
{
    const int p0 = scan_parts(P.kcap), pk = scan_parts(P.kcapr);
    return (int64_t)f * (p0 + P.NG * pk) + (r > 0 ? p0 + (r - 1) * pk : 0);
}

// Molecules per part of the rows' key counts (rows of several parts): block
// (part, row of the launch; the random groups of every frame, or the real pass)
__device__ __forceinline__ void b_scan_sums(KP P, Bufs B, int random, int bx_, int nbx_, int by_, int nby_)
{
    __shared__ int wsum[16];
    const int nr = random ? P.NG : 1, f = by_ / nr, r = random ? 1 + by_ - f * nr : 0;
    const int n = random ? P.kcapr : P.kcap, sp = scan_part(n);
    const int* c = B.mcnt + key_row(P, f, r);
    const int lo = bx_ * sp, hi = min(n, lo + sp);
    int t = 0;
    for (int i = lo + threadIdx.x; i < hi; i += blockDim.x) t += c[i];
    t = wave_incl_scan(t);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if (lane == 63) wsum[wid] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int w = 0; w < nw; w++) tot += wsum[w];
        B.msum[part_row(P, f, r) + bx_] = tot;
    }
}

__global__ void __launch_bounds__(1024) k_scan_sums(KP P, Bufs B, int random)
{
    b_scan_sums(P, B, random, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// Exclusive scan of the key counts of the real pass or the random groups of
// every frame (block (part, row)), each part starting from the molecules of
// the parts before it; writes the number of near molecules of the row
__device__ __forceinline__ void b_scan_rows(KP P, Bufs B, int random, int bx_, int nbx_, int by_, int nby_)
{
    __shared__ int wsum[16];
    __shared__ int carry;
    const int nr = random ? P.NG : 1, f = by_ / nr, r = random ? 1 + by_ - f * nr : 0;
    const int n = random ? P.kcapr : P.kcap, sp = scan_part(n);
    const int64_t row = (int64_t)f * (1 + P.NG) + r;
    const int* c = B.mcnt + key_row(P, f, r);
    int* st = B.mstart + key_row(P, f, r);
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    if (bx_ > 0 && wid == 0) {
        int t = 0;
        for (int k = lane; k < bx_; k += 64) t += B.msum[part_row(P, f, r) + k];
        t = wave_incl_scan(t);
        if (lane == 63) carry = t;
    }
    __syncthreads();
    // four consecutive keys per thread, the threads' sums scanned over the
    // wavefront (DPP) and across the block's wavefronts
    const int lo = bx_ * sp, hi = min(n, lo + sp);
    for (int base = lo; base < hi; base += 4 * blockDim.x) {
        const int i0 = base + 4 * threadIdx.x;
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = i0 + u < hi ? c[i0 + u] : 0;
        const int tsum = v[0] + v[1] + v[2] + v[3];
        const int incl = wave_incl_scan(tsum);
        if (lane == 63) wsum[wid] = incl;
        __syncthreads();
        int woff = 0, tot = 0;
        for (int w = 0; w < nw; w++) { if (w < wid) woff += wsum[w]; tot += wsum[w]; }
        int e = carry + woff + incl - tsum;
        // starts of empty keys are never read (the scatter reads the keys it
        // holds molecules of): most keys are empty, so only the others are written
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (i0 + u < hi && v[u] != 0) st[i0 + u] = e;
            e += v[u];
        }
        __syncthreads();
        if (threadIdx.x == 0) carry += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0 && hi == n) B.nnear[row] = carry;
}

__global__ void __launch_bounds__(1024) k_scan_rows(KP P, Bufs B, int random)
{
    b_scan_rows(P, B, random, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// molecules of the real pass or of the random groups sorted by key
__device__ __forceinline__ void b_mol_scatter(KP P, Bufs B, int random, int bx_, int nbx_, int by_, int nby_)
{
    // grid: x over a row's slots, y over the rows
    const int nr = random ? P.NG : 1;
    const int s = bx_ * blockDim.x + threadIdx.x;
    for (int fq = by_; fq < P.F * nr; fq += nby_) {
        const int f = fq / nr, grp = fq - (fq / nr) * nr;
        if (s >= (random ? group_slots(P, grp) : P.Mv)) continue;
        const int64_t row = row_base(P, f, random, grp);
        const int key = B.mkey[row + s];
        if (key < 0) continue;
        // the key's range starts where the scan put it; the molecule's rank
        // within the key was taken when the key was counted
        const int pos = B.mstart[key_row(P, f, random ? 1 + grp : 0) + key] + B.mrank[row + s];
        B.msorted[row + pos] = s;
    }
}

__global__ void k_mol_scatter(KP P, Bufs B, int random)
{
    b_mol_scatter(P, B, random, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// molecules of nv atoms that 64 lanes hold, one atom each
__host__ __device__ __forceinline__ int lane_molecules(int nv) { return 64 / nv; }

// Chunk offsets of the real pass or the random groups of every frame (one
// block), and the molecules per chunk.  A chunk costs some 3,000 instructions
// besides its distances (box, rows of cells, staging).  Near a compact solute its
// few hundred staged atoms outweigh them, and small chunks (P.mpt, P.mpt_r) have
// fewer; near an extended one (fewer than CHUNK_SPARSE solute atoms per cutoff^3
// of the volume that the near molecules fill) chunks of up to 512 atoms share
// them, as long as the launch keeps CHUNKS_REAL or CHUNKS_RANDOM chunks for its
// 4,096 wavefronts.  12,000 eight-atom molecules around a chain of 3,000 atoms
// (4.5 per cutoff^3), 20 frames: random passes 1,133 us with 16 molecules a chunk,
// 708 with 64; real pass 251 with 8, 169 with 18.  2,570 around a globule of 1,000
// (6.5), 12 frames of 10 passes: 504 us in all with 16, 574 with 55.
constexpr double CHUNK_SPARSE = 5.5;
constexpr int CHUNKS_REAL = 8192, CHUNKS_RANDOM = 4096;
// molecules per chunk that would leave a launch its chunks, were all of them near
__host__ __device__ __forceinline__ int64_t chunk_most(const KP& P, bool random)
{
    return (int64_t)P.F * (random ? P.K : 1) * P.Mv / (random ? CHUNKS_RANDOM : CHUNKS_REAL);
}
__host__ __device__ __forceinline__ bool chunks_vary(const KP& P)
{
    return P.mpt_auto && (chunk_most(P, false) > P.mpt || chunk_most(P, true) > P.mpt_r);
}

// (AUTO: for launches that chunks_vary lets choose; without, a microsecond less)
template <bool AUTO>
__device__ __forceinline__ void b_chunk_table(KP P, Bufs B, int random, int bx_, int nbx_, int by_, int nby_)
{
    __shared__ int wsum[16];
    __shared__ int carry;
    const int nr = random ? P.NG : 1, n = P.F * nr;
    int mpt = random ? P.mpt_r : P.mpt;
    if (AUTO && P.mpt_auto && chunk_most(P, random != 0) > mpt) {
        __shared__ double part[16];
        double t = 0.0;
        for (int idx = threadIdx.x; idx < n; idx += blockDim.x) {
            const int f = idx / nr, r = random ? 1 + idx - f * nr : 0;
            t += (double)B.nnear[(int64_t)f * (1 + P.NG) + r];
        }
        for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o, 64);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = t;
        __syncthreads();
        t = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) t += part[w];
        const double* H = B.geo[0].cell.H;
        const double vol = fabs(cm::cell_volume(H));
        const double dens = (double)P.nu * P.Mv * P.F * (random ? P.K : 1) / (vol * fmax(t, 1.0));
        if (dens * P.cutsys * P.cutsys * P.cutsys < CHUNK_SPARSE)
            mpt = max(mpt, min(min(64, 8 * lane_molecules(P.nv)), (int)(t / (random ? CHUNKS_RANDOM : CHUNKS_REAL))));
    }
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int base = 0; base < n; base += blockDim.x) {
        int idx = base + threadIdx.x;
        int v = 0;
        if (idx < n) {
            const int f = idx / nr, r = random ? 1 + idx - f * nr : 0;
            v = (B.nnear[(int64_t)f * (1 + P.NG) + r] + mpt - 1) / mpt;
        }
        const int incl = wave_incl_scan(v);
        if (lane == 63) wsum[wid] = incl;
        __syncthreads();
        int woff = 0, tot = 0;
        for (int w = 0; w < nw; w++) { if (w < wid) woff += wsum[w]; tot += wsum[w]; }
        if (idx < n) B.chunk_base[idx] = carry + woff + incl - v;
        __syncthreads();
        if (threadIdx.x == 0) carry += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        B.chunk_base[n] = carry;
        B.chunk_base[n + 1] = 0;   // the evaluation's chunk counter
        B.chunk_base[n + MPT_AT] = mpt;
    }
}

template <bool AUTO>
__global__ void __launch_bounds__(1024) k_chunk_table(KP P, Bufs B, int random)
{
    b_chunk_table<AUTO>(P, B, random, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// the molecule of frame f that a slot with the draw r is placed from
__device__ __forceinline__ int64_t slot_source(const KP& P, const Bufs& B, int f, uint32_t r)
{
    const int64_t lk = (int64_t)f * P.kb;
    const int nb = ldg(B.nbulk + lk);
    return nb > 0 ? (int64_t)ldg(B.blist + lk * P.Mv + cm::draw_index(r, nb)) : cm::draw_index(r, P.Mv);
}

// randomize_solvent! (src/mddf.jl:65-88), first half: the new centre of every
// slot; slots whose centre falls in a near cell get the Hilbert key of the (half-)cell
// (the others cannot have an atom within the cutoff of the solute)
__device__ __forceinline__ void b_place_keys(KP P, Bufs B, const unsigned* tab, int bx_, int nbx_, int by_, int nby_)
{
    // grid: x over the slots, y over the (frame, pass) pairs
    const int v = bx_ * blockDim.x + threadIdx.x;
    if (v >= P.Mv) return;
    for (int fk = by_; fk < P.F * P.K; fk += nby_) {
        const int f = fk / P.K;
        const int k = fk - f * P.K;
        const Geo g = ldc_geo(B.geo + f);
        const int grp = k / P.KM, sub = P.ksub;
        const int64_t e = row_base(P, f, true, grp) + (int64_t)(k - grp * P.KM) * P.Mv + v;
        cm::u32x4 r = cm::philox4x32_10({(uint32_t)v, (uint32_t)k, g.frame, cm::TAG_SLOT}, P.key0, P.key1);
        int c0, c1, c2;
        cell_of_draws(g, r.y, r.z, r.w, sub, c0, c1, c2);
        const int cell = ((c2 >> sub) * g.nc[1] + (c1 >> sub)) * g.nc[0] + (c0 >> sub);
        // (a copy of a molecule without a position has none)
        if (!B.near[(int64_t)f * P.cap + cell] ||
            (g.voids && (B.bflag[(int64_t)f * P.kb * P.Mv + slot_source(P, B, f, r.x)] & BULK_VOID))) {
            B.mkey[e] = -1;
            continue;
        }
        const int key = hilbert_key(tab, g.kbits + sub, c0, c1, c2);
        B.mkey[e] = key;
        B.mrank[e] = atomicAdd(&B.mcnt[key_row(P, f, 1 + grp) + key], 1);
    }
}

__global__ void k_place_keys(KP P, Bufs B)
{
    __shared__ unsigned tab[48];
    hilbert_load(tab);
    b_place_keys(P, B, tab, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// The random move of slot v of pass k (randomize_solvent!, src/mddf.jl:65-88):
// source molecule, new centre and turns
template <class TV>
struct SlotMove {
    const TV* x;
    double uc[3], ua[3];
    template <class GEO>
    __device__ SlotMove(const KP& P, const Bufs& B, const GEO& g, const TV* xv, int f, int k, int v)
    {
        const cm::u32x4 r = cm::philox4x32_10({(uint32_t)v, (uint32_t)k, g.frame, cm::TAG_SLOT}, P.key0, P.key1);
        const cm::u32x4 r2 = cm::philox4x32_10({(uint32_t)v, (uint32_t)k, g.frame, cm::TAG_SLOT + 1u}, P.key0, P.key1);
        x = xv + (int64_t)f * P.Nv * 3 + slot_source(P, B, f, r.x) * P.nv * 3;
        uc[0] = cm::u01(r.y); uc[1] = cm::u01(r.z); uc[2] = cm::u01(r.w);
        ua[0] = cm::u01(r2.x); ua[1] = cm::u01(r2.y); ua[2] = cm::u01(r2.z);
    }
};

// second half: the placement of the near slots, written in sorted order in
// fixed point.  Their FP64 positions are kept for verification only: k_resolve
// forms them again for the few molecules it looks at (72 of 120 bytes a water,
// in strided stores: 40,000 waters, 40 frames of 10 passes 282 us -> 171 us with
// the atoms of three-atom molecules read once; 8-atom molecules 601 -> 294 us).
template <class TV>
__device__ __forceinline__ void b_place_near(KP P, Bufs B, const TV* xv, int bx_, int nbx_, int by_, int nby_)
{
    // grid: x over the sorted positions of a group, y over the (frame, group) rows
    const int pos = bx_ * blockDim.x + threadIdx.x;
    for (int fg = by_; fg < P.F * P.NG; fg += nby_) {
        const int f = fg / P.NG;
        const int grp = fg - f * P.NG;
        if (pos >= ldg(B.nnear + (int64_t)f * (1 + P.NG) + 1 + grp)) continue;
        const int slot = ldg(B.msorted + row_base(P, f, true, grp) + pos);
        const int kk = slot / P.Mv, v = slot - kk * P.Mv, k = grp * P.KM + kk;
        const int64_t at = ((int64_t)f * P.K + (int64_t)grp * P.KM) * P.Nv + (int64_t)pos * P.nv;
        const Geo g = ldc_geo(B.geo + f);
        const SlotMove<TV> mv(P, B, g, xv, f, k, v);
        MolDstFix dst(B.P + 3 * at, B.vw_r + at, g, P.place_all != 0);
        // the placed centre is H uc (a rigid copy of a molecule of the frame):
        // the first atom's w carries the molecule's nearest-solute bound
        int cell, c0, c1, c2;
        cell_of_frac(g, mv.uc[0], mv.uc[1], mv.uc[2], cell, c0, c1, c2);
        const float ub = molecule_bound(g, bound_loads(P, B, g, f, cell, c0, c1, c2), c0, c1, c2, mv.uc);
        if (P.nv == 3) {
            cm::random_move(MolSrc3<TV>(mv.x), dst, 3, P.iref, g.cell, mv.uc, mv.ua);
        } else {
            cm::random_move(MolSrc<TV>(mv.x), dst, P.nv, P.iref, g.cell, mv.uc, mv.ua);
        }
        dst.set_w0(ub);
    }
}

template <class TV>
__global__ void __launch_bounds__(BLOCK) k_place_near(KP P, Bufs B, const TV* xv)
{
    b_place_near<TV>(P, B, xv, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// lexicographic minimum of two exact records, OR of the reference flags
__device__ __forceinline__ void rec_merge(Rec& r, const Rec& o)
{
    if (o.within && (!r.within || o.d < r.d || (o.d == r.d && (o.i < r.i || (o.i == r.i && o.j < r.j))))) {
        r.within = 1; r.i = o.i; r.j = o.j; r.d = o.d;
    }
    if (o.ref) { r.ref = 1; r.dref = fmin(r.dref, o.dref); }
}

__device__ __forceinline__ Rec rec_shfl_xor(const Rec& r, int o)
{
    Rec q;
    q.within = __shfl_xor(r.within, o, 64);
    q.i = __shfl_xor(r.i, o, 64);
    q.j = (int64_t)__shfl_xor((long long)r.j, o, 64);
    q.d = __shfl_xor(r.d, o, 64);
    q.ref = __shfl_xor(r.ref, o, 64);
    q.dref = __shfl_xor(r.dref, o, 64);
    return q;
}

// Matrix-core distances.  A tile is 16 staged solute atoms (rows) against one
// atom of 16 solvent molecules (columns): with s' = s - c and y' = y - c about
// the chunk centre c, v_mfma_f32_16x16x4_f32 forms |s'|^2 - 2 y'.s' for the 256
// pairs from the rows (s'x, s'y, s'z, |s'|^2) and the columns (-2 y', 1).  Lane
// l gives the component l / 16 of row and column l % 16 and receives rows
// 4 (l / 16) .. + 3 of its column.
typedef float f4m __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f4m pair_tile(float a, float b)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, f4m{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
}

// Running minimum b and second smallest s over four more values: the second
// smallest of {b <= s} and {x, y} is min(s, med3(b, x, y)), so each pair of
// values takes one three-input minimum and one median, and the medians go into
// s two at a time: five instructions for four values.
__device__ __forceinline__ void min2_4(float& b, float& s, const f4m& v)
{
    const float m = fminf(fminf(b, v[0]), v[1]), t0 = __builtin_amdgcn_fmed3f(b, v[0], v[1]);
    const float t1 = __builtin_amdgcn_fmed3f(m, v[2], v[3]);
    b = fminf(fminf(m, v[2]), v[3]);
    s = fminf(fminf(s, t0), t1);
}

// a minimum with its second smallest value and the code of its candidate
struct Min2 {
    float b, s;
    int c;
    __device__ __forceinline__ void init() { b = INFINITY; s = INFINITY; c = -1; }
    __device__ __forceinline__ void merge(float b2, float s2, int c2)
    {
        s = fminf(fmaxf(b, b2), fminf(s, s2));
        c = b2 < b ? c2 : c;
        b = fminf(b, b2);
    }
};

// The lanes 16 and 32 away hold the other rows of the same 16 molecules (per
// group): merged over them, lane l ends with molecule (l / 32) 16 + l % 16 of two
// groups or l % 16 of one.
template <int GH>
__device__ __forceinline__ Min2 gather_groups(const Min2 (&m)[GH], int lane)
{
    auto recv = [&](Min2& keep, const Min2& send, int o) {
        keep.merge(__shfl_xor(send.b, o, 64), __shfl_xor(send.s, o, 64), __shfl_xor(send.c, o, 64));
    };
    auto pick = [](bool hi, const Min2& x, const Min2& y) {
        Min2 r;
        r.b = hi ? y.b : x.b; r.s = hi ? y.s : x.s; r.c = hi ? y.c : x.c;
        return r;
    };
    const bool h5 = (lane & 32) != 0;
    Min2 k = GH == 2 ? pick(h5, m[0], m[GH - 1]) : m[0];
    recv(k, GH == 2 ? pick(h5, m[GH - 1], m[0]) : m[0], 32);
    recv(k, k, 16);
    return k;
}

// The same for four tiles of 16 columns: lane l ends with column l.
__device__ __forceinline__ Min2 gather_columns(const Min2* m, int lane)
{
    auto recv = [&](Min2& keep, const Min2& send, int o) {
        keep.merge(__shfl_xor(send.b, o, 64), __shfl_xor(send.s, o, 64), __shfl_xor(send.c, o, 64));
    };
    auto pick = [](bool hi, const Min2& x, const Min2& y) {
        Min2 r;
        r.b = hi ? y.b : x.b; r.s = hi ? y.s : x.s; r.c = hi ? y.c : x.c;
        return r;
    };
    const bool h4 = (lane & 16) != 0, h5 = (lane & 32) != 0;
    Min2 k0 = pick(h5, m[0], m[2]), k1 = pick(h5, m[1], m[3]);
    recv(k0, pick(h5, m[2], m[0]), 32);
    recv(k1, pick(h5, m[3], m[1]), 32);
    Min2 k = pick(h4, k0, k1);
    recv(k, pick(h4, k1, k0), 16);
    return k;
}

// LDS of the evaluation: the block's histograms, the launch's chunk table,
// then one area per wavefront
extern __shared__ float dyn[];

// LDS writes of a wavefront before reads of its other lanes (its LDS
// operations execute in order: only the compiler must keep them so)
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Column tiles: TQ solvent atoms of 16 G molecules each (TQ = 3: molecules of
// three atoms), or 16 G consecutive atoms (TQ = ATOMS: molecules of any size; G =
// 4 or 8)
constexpr int ATOMS = 0;
constexpr int EV_ROWS = 32;         // staged atoms per step (two row tiles)
constexpr int TCAP = 288;           // staged solute atoms per round (at least 256, a multiple of 32)
constexpr int SEG = 4;              // staging: consecutive atoms per lane

// words of a wavefront's area: staged components and indices, the columns of
// the tiles (-2 y' and |y'|^2 per atom), the segments of one step
__host__ __device__ constexpr int eval_wave_words(int G, int TQ) { return 5 * TCAP + 4 * (TQ == ATOMS ? 1 : TQ) * 16 * G + 2 * 64; }

// Block histograms.  Millions of records per launch go into a few hundred md
// and rdf bins: as global atomics they bounded the launch (the random passes of
// 40 frames of the globule job 1.65 ms with them, 1.05 ms with the same kernel
// and no md/rdf updates), so every block counts in LDS and adds its non-zero
// bins once at its end.  Word offsets into dyn; negative: straight to memory
// (histograms beyond EV_HIST words).
constexpr int EV_HIST = 8192;
struct EvHist {
    int md, rdf, gv;
    __host__ __device__ static int words(const KP& P)
    {
        return (2 * P.nbins <= EV_HIST ? 2 * P.nbins : 0) + gvw(P);
    }
    __host__ __device__ static int gvw(const KP& P)
    {
        const int64_t n = (int64_t)P.gnv * P.nbins;
        return 2 * P.nbins <= EV_HIST && n <= EV_HIST - 2 * P.nbins ? (int)n : 0;
    }
    __device__ explicit EvHist(const KP& P)
    {
        const bool in = 2 * P.nbins <= EV_HIST;
        md = in ? 0 : -1;
        rdf = in ? P.nbins : -1;
        gv = gvw(P) > 0 ? 2 * P.nbins : -1;
    }
};

__device__ __forceinline__ void ev_hist_clear(const KP& P)
{
    for (int k = threadIdx.x; k < EvHist::words(P); k += blockDim.x) ((unsigned*)dyn)[k] = 0u;
}

template <bool RANDOM>
__device__ __forceinline__ void ev_hist_flush(const KP& P, const Bufs& B)
{
    const EvHist h(P);
    const unsigned* sh = (const unsigned*)dyn;
    ull* md = RANDOM ? B.cnt_md_r : B.cnt_md;
    ull* rdf = RANDOM ? B.cnt_rdf_r : B.cnt_rdf;
    ull* gv = RANDOM ? B.cnt_gv_r : B.cnt_gv;
    if (h.md >= 0)
        for (int k = threadIdx.x; k < P.nbins; k += blockDim.x) {
            if (sh[k]) atomicAdd(&md[k], (ull)sh[k]);
            if (sh[P.nbins + k]) atomicAdd(&rdf[k], (ull)sh[P.nbins + k]);
        }
    const int n = EvHist::gvw(P);
    for (int k = threadIdx.x; k < n; k += blockDim.x)
        if (sh[h.gv + k]) atomicAdd(&gv[k], (ull)sh[h.gv + k]);
}

// The counts of a complete record (update_counters!, src/update_counters.jl:43-88)
// of solute atom i and atom `local` of the solvent molecule whose first atom is
// jbase (one solute molecule: i is molecule-local).  With h null, straight to
// memory.
template <bool RANDOM>
__device__ __forceinline__ void ev_hist_record(const KP& P, const Bufs& B, const EvHist* h, const Rec& r, int local, int64_t jbase)
{
    if (!r.within) return;
    const int b = r.bin;
    if (b >= P.nbins) return;   // unreachable: d <= cutoff (validated at job creation)
    unsigned* sh = (unsigned*)dyn;
    if (h && h->md >= 0) atomicAdd(&sh[h->md + b], 1u);
    else atomicAdd(&(RANDOM ? B.cnt_md_r : B.cnt_md)[b], 1ull);
    group_hit_local(RANDOM ? B.cnt_gu_r : B.cnt_gu, P.nbins, b, r.i, r.i, P.gu_ptr, P.gu_idx);
    if (h && h->gv >= 0) {
        if (!P.gv_ptr) atomicAdd(&sh[h->gv + local * P.nbins + b], 1u);
        else
            for (int k = P.gv_ptr[jbase + local]; k < P.gv_ptr[jbase + local + 1]; k++)
                atomicAdd(&sh[h->gv + P.gv_idx[k] * P.nbins + b], 1u);
    } else {
        group_hit_local(RANDOM ? B.cnt_gv_r : B.cnt_gv, P.nbins, b, local, jbase + local, P.gv_ptr, P.gv_idx);
    }
    if (r.ref && r.rbin < P.nbins) {
        if (h && h->rdf >= 0) atomicAdd(&sh[h->rdf + r.rbin], 1u);
        else atomicAdd(&(RANDOM ? B.cnt_rdf_r : B.cnt_rdf)[r.rbin], 1ull);
    }
}

// where a chunk of a launch lies: frame, random group, its row of the sorted
// molecules, first molecule, molecules, first atom (B.vw / B.vw_r, B.P)
struct ChunkAt {
    int f, grp, m0, nm, mpt;
    int64_t row, atom;
    template <class CB>
    __device__ ChunkAt(const KP& P, const Bufs& B, bool random, int ch, CB base)
    {
        const int nr = random ? P.NG : 1;
        mpt = chunk_molecules(P, B, random);
        int lo = 0, hi = P.F * nr;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (base(mid) <= ch) lo = mid; else hi = mid;
        }
        const int fq = __builtin_amdgcn_readfirstlane(lo);
        f = fq / nr;
        grp = fq - f * nr;
        m0 = __builtin_amdgcn_readfirstlane((ch - base(fq)) * mpt);
        row = row_base(P, f, random, grp);
        nm = min(mpt, ldg(B.nnear + (int64_t)f * (1 + P.NG) + (random ? 1 + grp : 0)) - m0);
        atom = (random ? ((int64_t)f * P.K + (int64_t)grp * P.KM) * P.Nv : (int64_t)f * P.Nv) + (int64_t)m0 * P.nv;
    }
};

// Minimum distances of the solvent molecules of one chunk, one wavefront.  The
// chunk's molecules are consecutive in the sorted order, so their atoms are
// contiguous.  Molecules of three atoms (TQ 3, at most 16 G of them): a column is
// a molecule, its three atoms are evaluated together.  Others: a column is an
// atom, and after the last round a lane holds one (two with eight tiles);
// molecules do not cross from one 64 lanes to the next.  (A column per molecule
// with four of its atoms at a time needs 16 molecules for full tiles: 16 of 40
// atoms are a box of half the solute.  5,000 solute atoms, 760 such molecules, 8
// frames of 10 passes: 2.60 ms so, 0.35 ms now, with the resolve.)  Records
// that FP32 decides are counted here; the molecules it cannot decide (a bin
// edge, the cutoff or dbulk within the guard, or an argmin closer than the
// guard) are left to k_resolve: one bit each in the chunk's word of resmask, and
// in the w of each atom the squared radius that holds its candidates, negative
// when it has none.
//
// What bounds it: per step of 32 staged atoms and 16 molecules a solvent atom
// costs two matrix instructions (64 cycles) and 12 vector ones (48 cycles) that
// keep the minimum, the second smallest and the step; they run side by side.
// The rest is latency (segment loads, LDS), which the block's other wavefronts
// fill: no FP64 here keeps the kernel at 128 registers, 16 wavefronts per CU.
template <class TU, class TV, bool RANDOM, int G, int TQ, bool VERIFY>
__device__ __forceinline__ void eval_chunk(const KP& P, const Bufs& B, const TU* xu, const TV* xv, int ch, const ChunkAt& at,
                                           int wofs, const EvHist& hist)
{
    // wofs: the wavefront's LDS area.  Staged atoms relative to the chunk
    // centre, atom n's component k (x, y, z, squared norm) at (n / 16) 64 + 16 k
    // + n % 16 (the order in which the lanes of a row tile read them), their
    // indices, the columns [atom of the block][-2 y'x, -2 y'y, -2 y'z, |y'|^2]
    // [molecule], the segments of a staging step
    constexpr bool FLAT = TQ == ATOMS;
    constexpr int MC = 16 * G;
    float* const lds = dyn + wofs;
    int* const si = (int*)(lds + 4 * TCAP);
    float* const yb = lds + 5 * TCAP;
    int2* const sd = (int2*)(yb + 4 * (FLAT ? 1 : TQ) * MC);
    // (opaque per chunk: what depends on the lane alone is formed where it is
    // used, not held in registers over the whole launch)
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    // groups are evaluated two at a time (half h of four groups: the lanes with
    // bit 4 equal to h keep its molecules)
    constexpr int GH = G == 1 ? 1 : 2;
    // the molecule of the chunk this lane decides, and whether it is the one
    // lane that does
    const int ml = (G == 4 ? ((lane >> 4) & 1) << 5 : 0) + (G == 1 ? 0 : (lane >> 5) << 4) + (lane & 15);
    const bool lead = G == 4 || (G == 2 ? (lane & 16) == 0 : lane < 16);
    const int f = at.f;
    const GeoC& g = *(const GeoC*)(B.geo + f);
    // FLAT: a block is once or twice 64 lanes, an atom each (molecules do not cross
    // from one 64 to the next): the lane's molecule in its 64, its atom there.  A
    // chunk of several blocks evaluates them one after the other from the same
    // staged atoms; where those do not fit the buffer, each block stages its own.
    constexpr int NL = G / 4 > 0 ? G / 4 : 1;
    const int mpl = FLAT ? lane_molecules(P.nv) : 0, apl = mpl * P.nv;
    const int lm = FLAT ? lane / P.nv : 0, la = lane - lm * P.nv;
    const int H = FLAT ? (at.nm + NL * mpl - 1) / (NL * mpl) : 1;
    unsigned long long um_ = 0;   // the molecules left open, one bit each in molecule order
    int h0 = 0, nb = H;
    while (h0 < H) {
        nb = FLAT ? min(nb, H - h0) : 1;
        const int mc = FLAT ? NL * h0 * mpl : 0, nm = FLAT ? min(at.nm - mc, NL * nb * mpl) : at.nm;   // molecules from mc on
        float4* vwb = (RANDOM ? B.vw_r : B.vw) + at.atom + mc * P.nv;   // their atoms
        const int na = nm * P.nv;
        const bool active = lead && ml < nm;
        const int slot = FLAT ? 0 : ldg(B.msorted + at.row + at.m0 + min(ml, nm - 1));
        // box of the atoms about one in their middle; the first atom's w is the
        // molecule's bound
        const gptr<const f4v> vg = (gptr<const f4v>)vwb;
        const f4v mid = vg[(nm >> 1) * P.nv];
        int cix = __builtin_amdgcn_readfirstlane(__float_as_int(mid.x)), ciy = __builtin_amdgcn_readfirstlane(__float_as_int(mid.y)),
            ciz = __builtin_amdgcn_readfirstlane(__float_as_int(mid.z));
        // position relative to the chunk's (integer) centre
        auto rel = [&](f4v y, float& x_, float& y_, float& z_) {
            fix_cart(g, __float_as_int(y.x) - cix, __float_as_int(y.y) - ciy, __float_as_int(y.z) - ciz, x_, y_, z_);
        };
        float alx = INFINITY, aly = INFINITY, alz = INFINITY, ahx = -INFINITY, ahy = -INFINITY, ahz = -INFINITY, um = 0.f;
        auto box = [&](const f4v& y) {
            float x_, y_, z_;
            rel(y, x_, y_, z_);
            alx = fminf(alx, x_); aly = fminf(aly, y_); alz = fminf(alz, z_);
            ahx = fmaxf(ahx, x_); ahy = fmaxf(ahy, y_); ahz = fmaxf(ahz, z_);
            um = fmaxf(um, y.w);
        };
        if (FLAT) {
            for (int e = lane; e < na; e += 256) {
                f4v y[4];
#pragma unroll
                for (int t = 0; t < 4; t++) y[t] = vg[min(e + 64 * t, na - 1)];
#pragma unroll
                for (int t = 0; t < 4; t++) box(y[t]);
            }
        } else {
            // 3-atom molecules: at most 3 G / 4 loads per lane, together
            f4v y[(3 * G + 3) / 4];
#pragma unroll
            for (int t = 0; t < (3 * G + 3) / 4; t++) y[t] = vg[min(64 * t + lane, na - 1)];
#pragma unroll
            for (int t = 0; t < (3 * G + 3) / 4; t++) box(y[t]);
        }
        um = wave_max(um);
        // the centre moves to the middle of the box (in whole units: exact), the
        // box with it (to FP32 rounding, inside the staging radius' slack)
        float bx, by, bz;   // half sides
        {
            const float lx = wave_min(alx), ly = wave_min(aly), lz = wave_min(alz);
            const float hx = wave_max(ahx), hy = wave_max(ahy), hz = wave_max(ahz);
            const float mx = 0.5f * (lx + hx), my = 0.5f * (ly + hy), mz = 0.5f * (lz + hz);
            bx = sgpr_f(0.5f * (hx - lx) + 1e-4f); by = sgpr_f(0.5f * (hy - ly) + 1e-4f); bz = sgpr_f(0.5f * (hz - lz) + 1e-4f);
            const float sc = ldexpf(1.0f, g.fix);
            cix += __builtin_amdgcn_readfirstlane((int)rintf((g.Hi32[0] * mx + g.Hi32[3] * my + g.Hi32[6] * mz) * sc));
            ciy += __builtin_amdgcn_readfirstlane((int)rintf((g.Hi32[1] * mx + g.Hi32[4] * my + g.Hi32[7] * mz) * sc));
            ciz += __builtin_amdgcn_readfirstlane((int)rintf((g.Hi32[2] * mx + g.Hi32[5] * my + g.Hi32[8] * mz) * sc));
        }
        const float rs_full = g.rstage;
        // Distances relative to the chunk centre c (a fixed-point position, no
        // rounding of its own): |y' - s'|^2 = (|s'|^2 - 2 y'.s') + |y'|^2.  With u =
        // 2^-24, Y >= |y'| and S >= |s'| for every staged atom, y' and s' are off by
        // at most rho u Y and rho u S (fix_cart), which moves d^2 by at most
        // 2 rho u (Y + S) d (d <= cutsys + 0.5 where it matters); the norms (3 u S^2,
        // 3 u Y^2), the four products and three additions of a tile in whatever
        // order (2 u Y S + 3 u (S^2 + 2 Y S)) and the last sum (u (Y + S)^2) add at
        // most 7 u (Y + S)^2.  Both widen the frame's guard for this chunk (FP32
        // here, every value rounded outward by the factors; S <= Y + the staging
        // radius, which is at most um + 0.3).  The columns hold -2 y' (exact scaling).
        float Gcf, cut2_hi_c, amb_c, gdir;   // gdir: the coordinates' rounding in a direct d^2, per d
        {
            const float Yb = __builtin_amdgcn_sqrtf(bx * bx + by * by + bz * bz) * (1.0f + 4e-6f) + 1e-3f;
            const float YS = 2.0f * Yb + fminf(rs_full, um + 0.3f) * (1.0f + 1e-5f) + 1e-3f;
            const float gd = 0x1p-24f * YS * (2.0f * g.rho * ((float)P.cutsys + 0.5f) + 7.0f * YS) * (1.0f + 1e-5f) + 1e-8f;
            gdir = sgpr_f((g.gd1 + 0x1p-23f * g.rho * YS) * (1.0f + 1e-5f));
            Gcf = sgpr_f((g.guard_up + gd) * (1.0f + 1e-6f));
            cut2_hi_c = sgpr_f((P.c2hi32 + Gcf) * (1.0f + 1e-6f));
            amb_c = sgpr_f(2.0f * Gcf + cut2_hi_c * 0x1p-20f);
        }
        // Staging radius.  Each molecule carries an upper bound U on its
        // atoms' nearest solute distance (molecule_bound).  A solute atom that
        // can decide anything for an atom p of the chunk (its FP64 nearest,
        // or within the FP32 decision band of it) is within
        // sqrt(U^2 + 2 G + amb) of p, hence of the AABB; staging out to
        // sqrt(U^2 + 2 amb + 4 G) plus a slack over FP32 rounding keeps every
        // such atom, and the farther ones cannot change a decision.
        float rs = rs_full;
        if (um < rs_full)
            rs = sgpr_f(fminf(rs_full, fminf(__builtin_amdgcn_sqrtf(fmaf(um, um, 2.0f * amb_c + 4.0f * Gcf)) * (1.0f + 1e-5f) + 1e-2f, um + 0.3f)));
        const float rs2 = rs * rs;
        int ilo[3], ihi[3];
        cell_range32(g, cix, ciy, ciz, bx + rs, by + rs, bz + rs, ilo, ihi);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            ilo[k] = __builtin_amdgcn_readfirstlane(ilo[k]);
            ihi[k] = __builtin_amdgcn_readfirstlane(ihi[k]);
        }
        const int ny = ihi[1] - ilo[1] + 1, nz = ihi[2] - ilo[2] + 1;
        const gptr<const int> st = (gptr<const int>)(B.start + (int64_t)f * (P.cap + 1));
        const gptr<const f4v> srt = (gptr<const f4v>)(B.sorted + (int64_t)f * B.nitems);
        // FLAT: the lane's atoms over all rounds: minimum, second smallest, its solute
        // atom and d^2 in the direct form
        float fb[NL], fs[NL], fd[NL];
        int fi[NL];
        // the lane's molecule over all rounds: minimum, second smallest and
        // argmin pair, and the same for the reference atom
        float mb = INFINITY, ms = INFINITY, rb = INFINITY, rsec = INFINITY;
        float mdir = INFINITY, rdir = INFINITY;   // the argmin pairs' d^2 in the direct form
        int mi = -1, ma = 0, ri = -1;
        const unsigned long long lt_mask = (1ull << lane) - 1ull;
        // The records of the lanes' molecules (`on`: slot and molecule m of the
        // chunk): minimum b, second smallest and argmin (solute atom i, atom a, d^2
        // in the direct form), and of the reference atom.  Returns whether FP32 leaves
        // the record open, and the squared radii w0 of every candidate's d^2 (FP32)
        // and w1 of the reference atom's.
        auto decide_record = [&](bool on, int slot_, int m, float b, float sec, int i, int a, float dir, float rb_, float rsec_,
                                 int ri_, float rdir_, float& w0, float& w1) {
            const int v = RANDOM ? slot_ - (slot_ / P.Mv) * P.Mv : slot_;   // solvent molecule (random passes: slot)
            const int64_t jbase = (int64_t)v * P.nv;
            Rec r = rec_zero();
            bool undec = false, amb = false;   // left to the FP64 resolve (amb: an argmin FP32 cannot separate)
            w0 = w1 = 0.f;
            if (on) {
                // a separated argmin decides with its direct d^2, whose guard shrinks
                // with d: fixed-point units (E) and the rounding of both positions
                // about the chunk centre, 2 rho u (Y + S) (gdir), times d, plus 2 rho + 4
                // units of d^2 and the roundings of decide32's own sums
                auto decide = [&](float d2, int& bn, int& bk) {
                    const float Gd = fmaf(g.gd2, d2, gdir * (__builtin_amdgcn_sqrtf(d2) * (1.0f + 1e-6f))) + g.gd0;
                    return decide32(P, Gd, d2, bn, bk);
                };
                int bn, bk;
                if (b <= cut2_hi_c) {
                    amb = !(sec - b > amb_c);
                    const int dd = decide(dir, bn, bk);
                    if (dd == 2) { r.within = 1; r.i = i; r.j = jbase + a; r.bin = bn; r.bulk = bk; }
                    undec = dd == 0;
                }
                if (rb_ <= cut2_hi_c) {
                    amb = amb || !(rsec_ - rb_ > amb_c);
                    const int dd = decide(rdir_, bn, bk);
                    if (dd == 2) { r.ref = 1; r.rbin = bn; }
                    undec = undec || dd == 0;
                }
                undec = undec || amb;
                if (undec) {
                    const float band = amb_c + 2.0f * Gcf;
                    w0 = fminf(b + band, cut2_hi_c);
                    w1 = fminf(fmaxf(rb_, b) + band, cut2_hi_c);
                } else {
                    ev_hist_record<RANDOM>(P, B, &hist, r, a, jbase);
                    if (!RANDOM && P.K > 0) B.bflag[(int64_t)f * P.kb * P.Mv + v] = inbulk(P, r) ? 1 : 0;
                    if constexpr (VERIFY) {
                        // verification: the record with its FP64 distances
                        auto dist = [&](int i_, int a_) {
                            double x0, x1, x2, y0, y1, y2;
                            load3(xu + (int64_t)f * P.Nu * 3, i_, x0, x1, x2);
                            if (RANDOM) load3(B.P + 3 * at.atom, (int64_t)m * P.nv + a_, y0, y1, y2);
                            else load3(xv + (int64_t)f * P.Nv * 3, jbase + a_, y0, y1, y2);
                            return sqrt(cm::canon_d2(B.geo[f].cell, x0, x1, x2, y0, y1, y2));
                        };
                        VRec o;
                        o.within = r.within; o.i = r.i; o.j = r.j; o.ref = r.ref; o.pad = 0;
                        o.d = r.within ? dist(r.i, a) : INFINITY;
                        o.dref = r.ref ? dist(ri_, P.iref) : INFINITY;
                        // slot: pass within the group times Mv plus the molecule
                        B.vrec[at.row + slot_] = o;
                    }
                }
            }
            return undec;
        };
        // the n staged atoms (FLAT: with block h, the first or last round of them)
        auto evaluate = [&](int n, int h, bool first, bool last) {
            const int nsteps = (n + EV_ROWS - 1) / EV_ROWS;
            if (h == 0) {
                // rows past n are far away and never the minimum
                if (lane < nsteps * EV_ROWS - n) {
                    const int q = n + lane, o = (q >> 4) * 64 + (q & 15);
                    lds[o] = 0.f; lds[o + 16] = 0.f; lds[o + 32] = 0.f; lds[o + 48] = 1e30f;
                    si[q] = -1;
                }
            }
            // the candidate of a code (step and rows): eight staged atoms, the
            // nearest of them (the tile's arithmetic is not repeated: when it
            // matters the minimum is below every other value by more than the
            // rounding of both forms, else the molecule is resolved in FP64)
            auto candidate = [&](int code, float yx, float yy, float yz, float& best) {
                const int k = (code >> 2) & 0x3fff, jl = code & 3;
                best = INFINITY;
                int bi = 0;
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const float* o = lds + k * 128 + t * 64 + 4 * jl;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float dx = yx - o[i], dy = yy - o[16 + i], dz = yz - o[32 + i];
                        const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
                        // (padding rows sit at the centre and are no candidates)
                        const bool lt = d2 < best && o[48 + i] < 1e29f;
                        best = lt ? d2 : best;
                        bi = lt ? k * EV_ROWS + t * 16 + 4 * jl + i : bi;
                    }
                }
                return si[bi];
            };
            if constexpr (FLAT) {
                const int mh = NL * h * mpl, left = nm - mh;   // the block's first molecule, molecules from there on
                auto on = [&](int k) { return lm < mpl && k * mpl + lm < left; };
                if (first) {
                    // the block's columns (zero where there is no atom)
#pragma unroll
                    for (int k = 0; k < NL; k++) {
                        float yx = 0.f, yy = 0.f, yz = 0.f;
                        if (on(k)) rel(vg[mh * P.nv + k * apl + lane], yx, yy, yz);
                        float* o = yb + k * 256 + lane;
                        o[0] = -2.0f * yx; o[64] = -2.0f * yy; o[128] = -2.0f * yz;
                        o[192] = fmaf(yx, yx, fmaf(yy, yy, yz * yz));
                        fb[k] = fs[k] = fd[k] = INFINITY;
                        fi[k] = -1;
                    }
                }
                wave_sync();
                float bc[G], vb[G], vs[G];
                int vc[G];
#pragma unroll
                for (int t = 0; t < G; t++) {
                    const float c = yb[(t >> 2) * 256 + (lane >> 4) * 64 + (t & 3) * 16 + (lane & 15)];
                    bc[t] = lane >= 48 ? 1.0f : c;
                    vb[t] = INFINITY; vs[t] = INFINITY; vc[t] = 0;
                }
#pragma unroll 1
                for (int k = 0; k < nsteps; k++) {
                    const float a0 = lds[k * 128 + lane], a1 = lds[k * 128 + 64 + lane];
#pragma unroll
                    for (int t = 0; t < G; t++) {
                        const f4m v0 = pair_tile(a0, bc[t]), v1 = pair_tile(a1, bc[t]);
                        const float b0 = vb[t];
                        min2_4(vb[t], vs[t], v0);
                        min2_4(vb[t], vs[t], v1);
                        vc[t] = vb[t] < b0 ? k : vc[t];
                    }
                }
#pragma unroll
                for (int k = 0; k < NL; k++) {
                    Min2 mt[4];
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        mt[t].b = vb[4 * k + t]; mt[t].s = vs[4 * k + t]; mt[t].c = (vc[4 * k + t] << 2) | (lane >> 4);
                    }
                    Min2 w = gather_columns(mt, lane);
                    const float* o = yb + k * 256 + lane;
                    w.b += o[192];
                    w.s += o[192];
                    if (w.b < fb[k]) fi[k] = candidate(w.c, -0.5f * o[0], -0.5f * o[64], -0.5f * o[128], fd[k]);
                    fs[k] = fminf(fmaxf(fb[k], w.b), fminf(fs[k], w.s));
                    fb[k] = fminf(fb[k], w.b);
                }
                if (last) {
#pragma unroll 1
                    for (int k = 0; k < NL; k++) {
                        const float b = k ? fb[NL - 1] : fb[0], sec = k ? fs[NL - 1] : fs[0], d = k ? fd[NL - 1] : fd[0];
                        const int is = k ? fi[NL - 1] : fi[0];
                        const bool has = on(k);
                        // the atoms of a molecule into its first lane (c: lane of the minimum);
                        // after the step with offset o a lane holds the next 2 o of its molecule
                        Min2 w;
                        w.b = has ? b : INFINITY; w.s = has ? sec : INFINITY; w.c = lane;
                        for (int o = 1; o < P.nv; o <<= 1) {
                            const float b2 = __shfl_down(w.b, o, 64), s2 = __shfl_down(w.s, o, 64);
                            const int c2 = __shfl_down(w.c, o, 64);
                            if (la + o < P.nv && lane + o < 64) w.merge(b2, s2, c2);
                        }
                        const int il = (lane + P.iref) & 63;
                        const int i = __shfl(is, w.c, 64), ri_ = __shfl(is, il, 64);
                        const float dir = __shfl(d, w.c, 64), rdir_ = __shfl(d, il, 64), rb_ = __shfl(b, il, 64), rsec_ = __shfl(sec, il, 64);
                        const int m = mc + mh + k * mpl + lm;   // of the chunk
                        const int slot_ = ldg(B.msorted + at.row + at.m0 + min(m, at.nm - 1));
                        float w0, w1;
                        const bool undec = decide_record(has && la == 0, slot_, m, w.b, w.s, i, w.c - lane, dir, rb_, rsec_, ri_, rdir_, w0, w1);
                        // the radius of every atom of the molecules left open
                        const int head = lane - la;
                        const float x0 = __shfl(w0, head, 64), x1 = __shfl(w1, head, 64);
                        if (__shfl(undec ? 1 : 0, head, 64) && has) {
                            const bool isref = la == P.iref;
                            const float wa = b <= x0 || (isref && b <= cut2_hi_c) ? (isref ? fmaxf(x0, x1) : x0) : -1.0f;
                            ((float*)(vwb + mh * P.nv + k * apl + lane))[3] = wa;
                        }
                        const int fl = __shfl(undec ? 1 : 0, (lane * P.nv) & 63, 64);
                        um_ |= __ballot(lane < mpl && fl != 0) << ((mc + mh + k * mpl) & 63);
                    }
                }
            } else {
                Min2 wm, wr;
                wm.init(); wr.init();
                // columns (zero where there is no molecule)
                for (int e = lane; e < MC * TQ; e += 64) {
                    const int m = e / TQ, qq = e - m * TQ;
                    float yx = 0.f, yy = 0.f, yz = 0.f;
                    if (m < nm) rel(vg[m * TQ + qq], yx, yy, yz);
                    float* o = yb + qq * 4 * MC + m;
                    o[0] = -2.0f * yx; o[MC] = -2.0f * yy; o[2 * MC] = -2.0f * yz;
                    o[3 * MC] = fmaf(yx, yx, fmaf(yy, yy, yz * yz));
                }
                wave_sync();
#pragma unroll 1
                for (int hh = 0; hh < G / GH; hh++) {
                    const float* yh = yb + hh * 16 * GH + (lane & 15);
                    float bc[GH][TQ], vb[GH][TQ], vs[GH][TQ];
                    int vc[GH][TQ];
#pragma unroll
                    for (int gg = 0; gg < GH; gg++)
#pragma unroll
                        for (int qq = 0; qq < TQ; qq++) {
                            const float c = yh[(qq * 4 + (lane >> 4)) * MC + gg * 16];
                            bc[gg][qq] = lane >= 48 ? 1.0f : c;
                            vb[gg][qq] = INFINITY; vs[gg][qq] = INFINITY; vc[gg][qq] = 0;
                        }
#pragma unroll 1
                    for (int k = 0; k < nsteps; k++) {
                        const float a0 = lds[k * 128 + lane], a1 = lds[k * 128 + 64 + lane];
#pragma unroll
                        for (int gg = 0; gg < GH; gg++)
#pragma unroll
                            for (int qq = 0; qq < TQ; qq++) {
                                const f4m v0 = pair_tile(a0, bc[gg][qq]), v1 = pair_tile(a1, bc[gg][qq]);
                                const float b0 = vb[gg][qq];
                                min2_4(vb[gg][qq], vs[gg][qq], v0);
                                min2_4(vb[gg][qq], vs[gg][qq], v1);
                                vc[gg][qq] = vb[gg][qq] < b0 ? k : vc[gg][qq];
                            }
                    }
                    // + |y'|^2, the atoms into the molecule; code: atom, step
                    Min2 mm[GH], mr[GH];
#pragma unroll
                    for (int gg = 0; gg < GH; gg++) {
                        mm[gg].init(); mr[gg].init();
#pragma unroll
                        for (int qq = 0; qq < TQ; qq++) {
                            const float y2 = yh[(qq * 4 + 3) * MC + gg * 16];
                            const float b2 = vb[gg][qq] + y2, s2 = vs[gg][qq] + y2;
                            const int code = (qq << 16) | (vc[gg][qq] << 2) | (lane >> 4);
                            mm[gg].merge(b2, s2, code);
                            if (qq == P.iref) { mr[gg].b = b2; mr[gg].s = s2; mr[gg].c = code; }
                        }
                    }
                    const Min2 gm = gather_groups<GH>(mm, lane), gr = gather_groups<GH>(mr, lane);
                    if (G < 4 || ((lane >> 4) & 1) == hh) { wm = gm; wr = gr; }
                }
                wave_sync();
                auto cand = [&](int code, float& best) {
                    float yx, yy, yz;
                    rel(vg[min(ml, nm - 1) * TQ + (code >> 16)], yx, yy, yz);
                    return candidate(code, yx, yy, yz, best);
                };
                if (wm.b < mb) { mi = cand(wm.c, mdir); ma = wm.c >> 16; }
                ms = fminf(fmaxf(mb, wm.b), fminf(ms, wm.s));
                mb = fminf(mb, wm.b);
                if (wr.b < rb) ri = cand(wr.c, rdir);
                rsec = fminf(fmaxf(rb, wr.b), fminf(rsec, wr.s));
                rb = fminf(rb, wr.b);
            }
            wave_sync();
        };
        // Staging walks rows of cells (x fastest in memory): a slot is the part
        // of one (y, z) row of the index box that lies in one periodic image
        // along x, so its atoms are one contiguous range of the sorted list.
        // With a diagonal cell, rows farther than rs from the AABB are
        // dropped and each row is trimmed to the x range within rs (plus a
        // slack over FP32 rounding); the per-atom AABB test below is exact.
        // The rows are cut into segments of up to SEG consecutive atoms; in a step
        // each lane takes one segment (listed in LDS by the rows' lanes), loads its
        // atoms together and appends the ones within rs of the AABB at
        // ballot/popcount offsets.  A step that would overflow the buffer evaluates
        // what is staged first.  The staged set does not depend on the order (FP32
        // ties between candidates go to the FP64 resolve).
        int q0;
        wrap_index(ilo[0], g.nc[0], q0);
        int q1;
        wrap_index(ihi[0], g.nc[0], q1);
        const int npc = q1 - q0 + 1;
        const int nslots = ny * nz * npc;
        // (slack over the FP32 rounding of absolute coordinates)
        const float slk = 1e-3f + 1e-6f * (fabsf(g.H32[0]) + fabsf(g.H32[4]) + fabsf(g.H32[8]));
        const float rsl = rs + slk, rsl2 = rsl * rsl;
        // (diagonal cells) the box's ends and the cells' sides
        const float hcx = g.H32[0] * __builtin_amdgcn_rcpf((float)g.nc[0]), hcy = g.H32[4] * __builtin_amdgcn_rcpf((float)g.nc[1]),
                    hcz = g.H32[8] * __builtin_amdgcn_rcpf((float)g.nc[2]), icx = __builtin_amdgcn_rcpf(hcx);
        const float ccx = g.Hfix[0] * (float)cix, ccy = g.Hfix[4] * (float)ciy, ccz = g.Hfix[8] * (float)ciz;
        bool split = false;
        int sb = -64, s0 = 0;   // slots of the current 64, its next segment
        int NS = 0;             // segments of the current 64 slots
        int cstart = 0, cnt = 0, nseg = 0, sexcl = 0, code = 0;   // the lane's row: atoms, segments, image
        for (bool first = true;; first = false) {
            int nst = 0;            // staged atoms (uniform)
            // (FLAT: the rows are formed again after an evaluation, which has no
            // registers to hold them)
            bool full = false, again = FLAT && !first;
            if (FLAT) { NS = 0; cstart = cnt = nseg = sexcl = code = 0; }
            for (;;) {
                while (again || (s0 >= NS && sb + 64 < nslots)) {
                    // the next 64 row slots
                    if (!again) { sb += 64; s0 = 0; }
                    again = false;
                    const int sl = sb + lane;
                    cstart = 0; cnt = 0;
                    if (sl < nslots) {
                        const int r = sl / npc, pc = sl - r * npc;
                        const int iy = ilo[1] + r % ny, iz = ilo[2] + r / ny;
                        int x0 = ilo[0], x1 = ihi[0];
                        bool keep = true;
                        if (g.ortho) {
                            const float dy = fmaxf(fabsf((iy + 0.5f) * hcy - ccy) - (by + 0.5f * hcy), 0.f);
                            const float dz = fmaxf(fabsf((iz + 0.5f) * hcz - ccz) - (bz + 0.5f * hcz), 0.f);
                            const float r2 = rsl2 - dy * dy - dz * dz;
                            if (r2 < 0.f) {
                                keep = false;
                            } else {
                                const float rx = __builtin_amdgcn_sqrtf(r2) * (1.0f + 1e-6f) + bx + slk;
                                x0 = max(x0, (int)floorf((ccx - rx) * icx - 1e-3f));
                                x1 = min(x1, (int)floorf((ccx + rx) * icx + 1e-3f));
                            }
                        }
                        const int mx = q0 + pc;
                        x0 = max(x0, mx * g.nc[0]);
                        x1 = min(x1, mx * g.nc[0] + g.nc[0] - 1);
                        if (keep && x0 <= x1) {
                            int my, mz;
                            const int cy = wrap_index(iy, g.nc[1], my), cz = wrap_index(iz, g.nc[2], mz);
                            const int crow = (cz * g.nc[1] + cy) * g.nc[0] - mx * g.nc[0];
                            cstart = st[crow + x0];
                            cnt = st[crow + x1 + 1] - cstart;
                            code = ((mx + 16) << 8) | ((my + 16) << 16) | ((mz + 16) << 24);
                        }
                    }
                    nseg = (cnt + SEG - 1) / SEG;
                    const int sincl = wave_incl_scan(nseg);
                    sexcl = sincl - nseg;
                    NS = __builtin_amdgcn_readlane(sincl, 63);
                    // (more than the buffer takes, before any is staged: about half of
                    // the rows' atoms pass the test of the box)
                    if (FLAT && nb > 1 && NS * SEG > 2 * TCAP) split = true;
                    if (split) break;
                }
                if (split || s0 >= NS) break;
                f4v q[SEG];
                bool pass[SEG];
                int total = 0;
                // segments s0 .. s0 + 63: first atom, row lane and atoms
                for (int t = max(0, s0 - sexcl); t < nseg && sexcl + t < s0 + 64; t++)
                    sd[sexcl + t - s0] = make_int2(cstart + SEG * t, code | min(SEG, cnt - SEG * t));
                wave_sync();
                int2 d = sd[lane];
                wave_sync();
                if (s0 + lane >= NS) d = make_int2(0, 0);
                const int n = d.y & 255;
#pragma unroll
                for (int u = 0; u < SEG; u++) q[u] = srt[u < n ? d.x + u : 0];
                // the image's origin relative to the centre
                const int ox = ((((d.y >> 8) & 255) - 16) << g.fix) - cix, oy = ((((d.y >> 16) & 255) - 16) << g.fix) - ciy,
                          oz = ((((d.y >> 24) & 255) - 16) << g.fix) - ciz;
#pragma unroll
                for (int u = 0; u < SEG; u++) {
                    float x_, y_, z_;
                    fix_cart(g, __float_as_int(q[u].x) + ox, __float_as_int(q[u].y) + oy, __float_as_int(q[u].z) + oz, x_, y_, z_);
                    q[u].x = x_; q[u].y = y_; q[u].z = z_;
                    const float dx = fmaxf(fabsf(q[u].x) - bx, 0.f), dy = fmaxf(fabsf(q[u].y) - by, 0.f),
                                dz = fmaxf(fabsf(q[u].z) - bz, 0.f);
                    pass[u] = u < n && dx * dx + dy * dy + dz * dz <= rs2;
                    total += __popcll(__ballot(pass[u]));
                }
                full = nst + total > TCAP;
                if (full) break;
                s0 += 64;
#pragma unroll
                for (int u = 0; u < SEG; u++) {
                    const unsigned long long m = __ballot(pass[u]);
                    if (pass[u]) {
                        const int a = nst + __popcll(m & lt_mask);
                        const int o = (a >> 4) * 64 + (a & 15);
                        lds[o] = q[u].x; lds[o + 16] = q[u].y; lds[o + 32] = q[u].z;
                        lds[o + 48] = fmaf(q[u].x, q[u].x, fmaf(q[u].y, q[u].y, q[u].z * q[u].z));
                        si[a] = __float_as_int(q[u].w);
                    }
                    nst += __popcll(m);
                }
            }
            if (full && nb > 1) split = true;
            if (split) break;
            if (FLAT || nst > 0) {
#pragma unroll 1
                for (int h = 0; h < nb; h++) evaluate(nst, h, first, !full);
            }
            if (!full) break;
        }
        if (split) {
            nb = 1;
            continue;
        }
        h0 += nb;
        if constexpr (!FLAT) {
            float w0, w1;
            const bool undec = decide_record(active, slot, ml, mb, ms, mi, ma, mdir, rb, rsec, ri, rdir, w0, w1);
            if (undec) {
                float* o = (float*)(vwb + ml * TQ);
#pragma unroll
                for (int q = 0; q < TQ; q++) o[4 * q + 3] = q == P.iref ? fmaxf(w0, w1) : w0;
            }
            um_ = __ballot(undec);
            if (G == 2) um_ = (um_ & 0xffffull) | ((um_ >> 16) & 0xffff0000ull);
            if (G == 4) um_ = (um_ & 0xffff00000000ffffull) | ((um_ & 0xffff0000ull) << 16) | ((um_ >> 16) & 0xffff0000ull);
        }
    }
    if (lane == 0) {
        if (at.mpt > 32) ((ull*)B.resmask)[ch] = um_;
        else B.resmask[ch] = (unsigned)um_;
        if (um_) atomicAdd(&B.stats[0], (ull)__popcll(um_));
    }
}

// Chunks of one job's launch, handed to the wavefronts (w of the launch's W):
// w, w + W, ... below tdyn, then (with a counter ctr, zero at the start of the
// launch) the chunks from tdyn on in the order the wavefronts ask for them, so
// the ones that finish early take more of the last chunks.  The chunks' costs
// vary with their staged atoms, and a fixed stride alone leaves a tail of
// wavefronts still busy; requests go to one device-wide counter, so only the
// last DYN_PCT per cent are handed out that way, a few consecutive chunks per
// request.
struct ChunkFeed {
    int total, W, tdyn, dgrab, dnext, dend;
    int* ctr;
    __device__ ChunkFeed(int total_, int W_, int* ctr_) : total(total_), W(W_), dnext(0), dend(0), ctr(ctr_)
    {
        const int ndyn = (int)((int64_t)total * DYN_PCT / 100);
        tdyn = total >= DYN_MIN * W ? total - ndyn : total;
        dgrab = max(1, ndyn / (W * DYN_GRABS));
    }
    // the chunk to run given the next one of the stride
    __device__ int next(int c)
    {
        if (c < tdyn || tdyn == total) return c;
        if (dnext < dend) return dnext++;
        int g = 0;
        if ((threadIdx.x & 63) == 0) g = atomicAdd(ctr, dgrab);
        dnext = tdyn + __builtin_amdgcn_readfirstlane(g);
        dend = dnext + dgrab;
        return dnext++;
    }
};

// A kernel's first two arguments (KP, Bufs) read again from the kernel argument
// segment: called per chunk, so that the compiler loads a field where it is
// used (a scalar cache hit) instead of holding them all in scalar registers
// over the whole launch (about a hundred spilled to vector registers otherwise).
struct JobArgs {
    const KP& P;
    const Bufs& B;
};
__device__ __forceinline__ JobArgs job_args()
{
    using cptr = __attribute__((address_space(4))) const char*;
    cptr k = (cptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    constexpr size_t off = (sizeof(KP) + alignof(Bufs) - 1) / alignof(Bufs) * alignof(Bufs);
    return {*(const KP*)k, *(const Bufs*)(k + off)};
}

// Evaluation of one job's launch (persistent grid, blocks of independent
// wavefronts that share the LDS histograms and the chunk table)
template <class TU, class TV, bool RANDOM, int G, int TQ, bool VERIFY>
__global__ void __launch_bounds__(1024) k_eval_tiles(KP P, Bufs B, const TU* xu, const TV* xv)
{
    const int nfp = P.F * (RANDOM ? P.NG : 1);
    const bool cb_lds = nfp + 1 <= CBCAP;
    int* cbs = (int*)dyn + EvHist::words(P);
    const int wbase = (EvHist::words(P) + (cb_lds ? nfp + 1 : 0) + 3) & ~3;
    if (cb_lds)
        for (int k = threadIdx.x; k <= nfp; k += blockDim.x) cbs[k] = B.chunk_base[k];
    ev_hist_clear(P);
    __syncthreads();
    const EvHist hist(P);
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    const int total = B.chunk_base[nfp];
    ChunkFeed feed(total, gridDim.x * nw, B.chunk_base + nfp + 1);
    auto base = [&](int k) { return cb_lds ? cbs[k] : B.chunk_base[k]; };
    for (int ch = feed.next(blockIdx.x + wid * gridDim.x); ch < total; ch = feed.next(ch + feed.W)) {
        const JobArgs a = job_args();
        const ChunkAt at(a.P, a.B, RANDOM, ch, base);
        eval_chunk<TU, TV, RANDOM, G, TQ, VERIFY>(a.P, a.B, xu, xv, ch, at, wbase + wid * eval_wave_words(G, TQ), hist);
    }
    __syncthreads();
    ev_hist_flush<RANDOM>(P, B);
}

// FP64 records of the molecules FP32 left undecided: a block takes a few
// consecutive chunks of a row, lists their marked molecules in LDS and gives each
// 16 lanes.  They walk the rows of cells within reach of the atoms that the
// evaluation left a radius (of molecules of other than three atoms usually one or
// two: the others are farther than the minimum by more than the guard).  Every
// solute atom within the radius (FP32, wider than the guard) is evaluated exactly,
// ties to the smallest (i, j).  Kept out of the evaluation, whose registers and
// code it would double.
constexpr int RES_CHUNKS = 64;

// chunks a block of the resolve takes at a time: 64, in small launches as few
// as give about a thousand blocks (34 frames of 50 chunks of ureas: 67 us a launch
// with a block a frame, 55 so)
__host__ __device__ __forceinline__ int64_t resolve_row_chunks(const KP& P, bool random)
{
    const int64_t mpt = random ? P.mpt_r : P.mpt;
    return ((random ? (int64_t)P.KM : 1) * P.Mv + mpt - 1) / mpt;
}
__host__ __device__ __forceinline__ int resolve_step(const KP& P, bool random)
{
    const int64_t n = resolve_row_chunks(P, random) * P.F * (random ? P.NG : 1) / 1024;
    return n < 2 ? 2 : (n > RES_CHUNKS ? RES_CHUNKS : (int)n);
}

// cm::random_move of slot v of pass k by 16 lanes (sub), atoms at a stride: the
// same operations in the same order, so the same positions (FP64, at yp).  Every
// lane forms the centre, from the wrapped positions the others left there.
template <class TV>
__device__ __forceinline__ void place_by_lanes(const KP& P, const Bufs& B, const TV* xv, int f, int k, int v, double* yp, int sub)
{
    const cm::Cell64& c = B.geo[f].cell;
    const SlotMove<TV> mv(P, B, B.geo[f], xv, f, k, v);
    const MolSrc<TV> x(mv.x);
    const double rx = x(P.iref, 0), ry = x(P.iref, 1), rz = x(P.iref, 2);
    for (int a = sub; a < P.nv; a += 16) {
        double ox, oy, oz;
        cm::minimage(c, x(a, 0) - rx, x(a, 1) - ry, x(a, 2) - rz, &ox, &oy, &oz);
        yp[3 * a] = rx + ox; yp[3 * a + 1] = ry + oy; yp[3 * a + 2] = rz + oz;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
    double cx = 0.0, cy = 0.0, cz = 0.0;
    for (int a = 0; a < P.nv; a++) { cx += yp[3 * a]; cy += yp[3 * a + 1]; cz += yp[3 * a + 2]; }
    cx = cx / (double)P.nv; cy = cy / (double)P.nv; cz = cz / (double)P.nv;
    const double* H = c.H;
    const double n0 = H[0] * mv.uc[0] + H[3] * mv.uc[1] + H[6] * mv.uc[2];
    const double n1 = H[1] * mv.uc[0] + H[4] * mv.uc[1] + H[7] * mv.uc[2];
    const double n2 = H[2] * mv.uc[0] + H[5] * mv.uc[1] + H[8] * mv.uc[2];
    double A[9];
    cm::eulermat_turns(mv.ua[0], mv.ua[1], mv.ua[2], A);
    // (every lane has read the wrapped positions before one replaces them)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
    for (int a = sub; a < P.nv; a += 16) {
        const double dx = yp[3 * a] - cx, dy = yp[3 * a + 1] - cy, dz = yp[3 * a + 2] - cz;
        yp[3 * a] = A[0] * dx + A[1] * dy + A[2] * dz + n0;
        yp[3 * a + 1] = A[3] * dx + A[4] * dy + A[5] * dz + n1;
        yp[3 * a + 2] = A[6] * dx + A[7] * dy + A[8] * dz + n2;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
}

template <class TU, class TV, bool RANDOM, bool VERIFY>
__device__ __forceinline__ void resolve_one(const KP& P, const Bufs& B, const TU* xu, const TV* xv, int f, int grp, int64_t row,
                                            int64_t atom, int pos)
{
    // pos: sorted position in the row (the same in the 16 lanes), -1: none
    const int lane = threadIdx.x & 63, sub = lane & 15;
    const GeoC& g = *(const GeoC*)(B.geo + f);
    Rec r = rec_zero();
    int64_t v = 0, jbase = 0;
    int slot = 0;
    if (pos >= 0) {
        const gptr<const f4v> vg = (gptr<const f4v>)((RANDOM ? B.vw_r : B.vw) + atom + (int64_t)pos * P.nv);
        const gptr<const int> st = (gptr<const int>)(B.start + (int64_t)f * (P.cap + 1));
        const gptr<const f4v> srt = (gptr<const f4v>)(B.sorted + (int64_t)f * B.nitems);
        const TU* xuf = xu + (int64_t)f * P.Nu * 3;
        slot = ldg(B.msorted + row + pos);
        v = RANDOM ? slot - (slot / P.Mv) * P.Mv : slot;
        jbase = v * P.nv;
        double* const yp = B.P + 3 * (atom + (int64_t)pos * P.nv);
        if (RANDOM && !P.place_all) {
            // the molecule's FP64 positions (k_place_near's move): few atoms by one
            // lane, more by all
            const int pass = grp * P.KM + slot / P.Mv;
            if (P.nv > 4) {
                place_by_lanes(P, B, xv, f, pass, (int)v, yp, sub);
            } else {
                if (sub == 0) {
                    MolDst64 dst(yp);
                    const SlotMove<TV> mv(P, B, B.geo[f], xv, f, pass, (int)v);
                    cm::random_move(MolSrc<TV>(mv.x), dst, P.nv, P.iref, B.geo[f].cell, mv.uc, mv.ua);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
                __builtin_amdgcn_wave_barrier();
            }
        }
        for (int ab = 0; ab < P.nv; ab += 16) {
            const float wl = ab + sub < P.nv ? vg[ab + sub].w : -1.0f;
            unsigned open = (unsigned)(__ballot(wl >= 0.0f) >> (lane & 48)) & 0xffffu;
            while (open) {
                // four, two or one of the open atoms at a time, `w` lanes each
                const int left = __popc(open), w = left > 2 ? 4 : (left == 2 ? 8 : 16), wl0 = sub & (w - 1);
                unsigned mine = open;
                for (int q = 0; q < 16 / w; q++) {
                    if (q < sub / w) mine &= mine - 1u;
                    open &= open - 1u;
                }
                if (!mine) continue;
                const int a = ab + __builtin_ctz(mine);
                const f4v y = vg[a];
                const bool isref = a == P.iref;
                const float R2 = y.w;
                double y0, y1, y2;
                if (RANDOM) load3((const double*)yp, a, y0, y1, y2);
                else load3(xv + (int64_t)f * P.Nv * 3, jbase + a, y0, y1, y2);
                const int ux = __float_as_int(y.x), uy = __float_as_int(y.y), uz = __float_as_int(y.z);
                const float rr_ = __builtin_amdgcn_sqrtf(R2) * (1.0f + 1e-5f) + 1e-3f;
                int jlo[3], jhi[3];
                cell_range32(g, ux, uy, uz, rr_, rr_, rr_, jlo, jhi);
                const int nyr = jhi[1] - jlo[1] + 1, rows = nyr * (jhi[2] - jlo[2] + 1);
                for (int rr = wl0; rr < rows; rr += w) {
                    int my, mz;
                    const int cy = wrap_index(jlo[1] + rr % nyr, g.nc[1], my), cz = wrap_index(jlo[2] + rr / nyr, g.nc[2], mz);
                    const int crow = (cz * g.nc[1] + cy) * g.nc[0];
                    for (int x0 = jlo[0]; x0 <= jhi[0];) {
                        // the part of the row in one periodic image
                        int mx;
                        const int cx = wrap_index(x0, g.nc[0], mx);
                        const int nx = min(jhi[0] - x0 + 1, g.nc[0] - cx);
                        const int qx = ux - (mx << g.fix), qy = uy - (my << g.fix), qz = uz - (mz << g.fix);
                        const int k1 = st[crow + cx + nx];
                        for (int k = st[crow + cx]; k < k1; k += 8) {
                            f4v s[8];
#pragma unroll
                            for (int u = 0; u < 8; u++) s[u] = srt[min(k + u, k1 - 1)];
#pragma unroll
                            for (int u = 0; u < 8; u++) {
                                float dx, dy, dz;
                                fix_cart(g, __float_as_int(s[u].x) - qx, __float_as_int(s[u].y) - qy, __float_as_int(s[u].z) - qz,
                                         dx, dy, dz);
                                if (k + u < k1 && fmaf(dx, dx, fmaf(dy, dy, dz * dz)) <= R2) {
                                    const int i = __float_as_int(s[u].w);
                                    double p0, p1, p2;
                                    load3(xuf, i, p0, p1, p2);
                                    const double d2 = cm::canon_d2(B.geo[f].cell, p0, p1, p2, y0, y1, y2);
                                    if (d2 <= P.cut2) rec_offer(r, i, jbase + a, sqrt(d2), isref);
                                }
                            }
                        }
                        x0 += nx;
                    }
                }
            }
        }
    }
    for (int o = 8; o >= 1; o >>= 1) rec_merge(r, rec_shfl_xor(r, o));
    if (pos >= 0 && sub == 0) {
        rec_complete(P, r);
        ev_hist_record<RANDOM>(P, B, nullptr, r, (int)(r.j - jbase), jbase);
        if (!RANDOM && P.K > 0) B.bflag[(int64_t)f * P.kb * P.Mv + v] = inbulk(P, r) ? 1 : 0;
        if constexpr (VERIFY) {
            VRec o;
            o.within = r.within; o.i = r.i; o.j = r.j; o.d = r.d; o.ref = r.ref; o.pad = 0; o.dref = r.dref;
            B.vrec[row + slot] = o;
        }
    }
}

// grid: x over the parts of a row (resolve_step chunks each), y over the rows
template <class TU, class TV, bool RANDOM, bool VERIFY>
__device__ __forceinline__ void b_resolve(const KP& P, const Bufs& B, const TU* xu, const TV* xv, int bx_, int nbx_, int by_,
                                          int nby_)
{
    __shared__ int list[RES_CHUNKS * 64];
    __shared__ int nlist;
    const int nr = RANDOM ? P.NG : 1, mpt = chunk_molecules(P, B, RANDOM), step = resolve_step(P, RANDOM);
    for (int fq = by_; fq < P.F * nr; fq += nby_) {
        const int f = fq / nr, grp = fq - f * nr;
        const int c0 = ldg(B.chunk_base + fq), c1 = ldg(B.chunk_base + fq + 1);
        const int64_t row = row_base(P, f, RANDOM, grp);
        const int64_t atom = RANDOM ? ((int64_t)f * P.K + (int64_t)grp * P.KM) * P.Nv : (int64_t)f * P.Nv;
        for (int cb = c0 + bx_ * step; cb < c1; cb += nbx_ * step) {
            // one wavefront lists the marked molecules' positions
            if (threadIdx.x < 64) {
                const int ch = cb + threadIdx.x;
                ull m = (int)threadIdx.x < step && ch < c1 ? (mpt > 32 ? ((const ull*)B.resmask)[ch] : B.resmask[ch]) : 0ull;
                const int n = __popcll(m), incl = wave_incl_scan(n);
                int o = incl - n;
                while (m) {
                    list[o++] = (ch - c0) * mpt + __ffsll((long long)m) - 1;
                    m &= m - 1ull;
                }
                if (threadIdx.x == 63) nlist = incl;
            }
            __syncthreads();
            const int n = nlist;
            for (int k = 0; k < n; k += BLOCK / 16) {
                const int q = k + (threadIdx.x >> 4);
                resolve_one<TU, TV, RANDOM, VERIFY>(P, B, xu, xv, f, grp, row, atom, q < n ? list[q] : -1);
            }
            __syncthreads();
        }
    }
}

template <class TU, class TV, bool RANDOM, bool VERIFY>
__global__ void __launch_bounds__(BLOCK, 3) k_resolve(KP P, Bufs B, const TU* xu, const TV* xv)
{
    b_resolve<TU, TV, RANDOM, VERIFY>(P, B, xu, xv, blockIdx.x, gridDim.x, blockIdx.y, gridDim.y);
}

// parts of the resolve's grid along a row: about 2048 blocks in all, at most
// one per step of chunks
int64_t resolve_parts(const KP& P, bool random)
{
    const int64_t rows = (int64_t)P.F * (random ? P.NG : 1), step = resolve_step(P, random);
    return std::max<int64_t>(1, std::min<int64_t>((resolve_row_chunks(P, random) + step - 1) / step, 2048 / rows + 1));
}

// ---------------------------------------------------------------------------
// molecule pairs on the matrix cores (molecules of up to CL_ATOMS atoms)
// ---------------------------------------------------------------------------
// Solute molecules, sorted along a Hilbert curve, fill the 16 rows of A tiles:
// RPM rows per molecule (1 where both sides are single atoms, else 4, 8 or 16),
// 16 / RPM molecules per tile; solvent
// molecules in the same kind of order fill the 16 columns of B clusters, one
// column tile per atom.  Positions are FP32 relative to the tile's (cluster's)
// fixed-point centre.  A wavefront takes one B cluster and every A tile whose box
// is within the cutoff of its box: one matrix instruction per solvent atom q
// gives 256 distances, four per lane, so a lane holds one molecule pair (RPM 4),
// a part of one, or four of single atoms, and keeps its minimum, second smallest
// value and the minima over the reference atoms.  The pairs within the cutoff
// (about one in six) go to an LDS queue and are counted 64 at a time; the ones FP32
// cannot decide go on to a second queue and are formed again in FP64, 64 at a time,
// the last of a wavefront's with the lanes shared out among them.  Where the
// clusters are fewer than the wavefronts, S of these share one, its tiles in turn.
//
// The cell walk evaluates a pair in one thread, some 25 vector instructions per
// distance with the tests of its neighbourhood; here a distance costs 2.25 (its
// code, minimum and second smallest), and everything per tile or per pair
// within the cutoff is shared by 64 lanes.  Measured, real pass: 33,400 waters
// in a 100 A box, 24 frames, 3.66 -> 2.60 ms; 12,000 ureas in a triclinic 90 A
// cell, 20 frames, 3.45 -> 2.63 ms; 901 waters, 40 frames, 0.76 -> 0.19 ms.
// Bound by vector issue (busy 64 % of the time on the first, the matrix cores
// 21 %, four wavefronts per SIMD at 128 registers).  Tiles hold few molecules
// and the clusters 16 because the pairs of two boxes in reach, but not of
// their molecules, are the waste: five of six here.
constexpr int CL_ATOMS = 16;     // largest molecules of these kernels
constexpr int CL_SUP = 16;       // A tiles per super tile (the unit of the first box test)
constexpr int CL_Q = 128;        // queue entries per wavefront
constexpr int CL_WORDS = 5 * CL_Q + 2 * CL_Q + 256;   // LDS words per wavefront: pair queue, deferred pairs, tile centres
constexpr unsigned CL_DRAWN = 0x80000000u;            // (molecule indices are below 2^31)

// k_cl_eval's arguments as they lie in the kernel argument segment
template <class TU, class TV>
struct ClArgs {
    KP P;
    Bufs B;
    const TU* xu;
    const TV* xv;
    int S, Sg;
};

// Sort key of a molecule, the 2^bits grid cell of its centre, and the largest
// molecule radius of a frame (blockIdx.y: frame, blockIdx.z: side).  The centre
// is kept for k_cl_build: a molecule sorted by one periodic image and built at
// another would span its tile across the cell.
template <class T>
__global__ void __launch_bounds__(BLOCK) k_cl_keys(KP P, Bufs B, const T* xu, const T* xv)
{
    __shared__ unsigned tab[48];
    hilbert_load(tab);
    const int side = blockIdx.z, f = blockIdx.y;
    const ClSide s = B.cl[side];
    Geo& g = B.geo[f];
    const T* x = (side ? xv : xu) + (int64_t)f * s.M * s.n * 3;
    float r2 = 0.f;
    for (int m = blockIdx.x * blockDim.x + threadIdx.x; m < s.M; m += gridDim.x * blockDim.x) {
        const int64_t a0 = (int64_t)m * s.n;
        double c[3], fr[3], n[3], x0, y0, z0;
        mol_centre(g, x, a0, s.n, c);
        wrap_point(g, c[0], c[1], c[2], fr, n);
        const int top = (1 << s.bits) - 1;
        int ck[3];
        for (int k = 0; k < 3; k++) ck[k] = min(top, max(0, (int)(fr[k] * (top + 1))));
        const int key = hilbert_key(tab, s.bits, ck[0], ck[1], ck[2]);
        const int64_t it = (int64_t)f * s.M + m;
        for (int k = 0; k < 3; k++) s.cen[3 * it + k] = c[k];
        s.key[it] = key;
        s.rank[it] = atomicAdd(&s.cnt[((int64_t)f << (3 * s.bits)) + key], 1);
        load3(x, a0, x0, y0, z0);
        for (int a = 0; a < s.n; a++) {
            double xa, ya, za;
            load3(x, a0 + a, xa, ya, za);
            float ox, oy, oz;
            minimage32(g, (float)(xa - x0), (float)(ya - y0), (float)(za - z0), ox, oy, oz);
            const float dx = ox - (float)(c[0] - x0), dy = oy - (float)(c[1] - y0), dz = oz - (float)(c[2] - z0);
            r2 = fmaxf(r2, dx * dx + dy * dy + dz * dz);
        }
    }
    const float r = block_max(r2 > 0.f || blockIdx.x * blockDim.x + threadIdx.x < s.M ? sqrtf(r2) * 1.0001f + 1e-3f : 0.f);
    // (self: both radii)
    radii_report(P, B, 1, f, side == 0 ? r : 0.f, side == 1 || P.self_ ? r : 0.f, gridDim.x * gridDim.z);
}

// exclusive scan of the key counts, one block per frame and side
__global__ void __launch_bounds__(1024) k_cl_scan(KP P, Bufs B)
{
    __shared__ int wsum[16];
    __shared__ int carry;
    const ClSide s = B.cl[blockIdx.y];
    const int n = 1 << (3 * s.bits);
    const int* c = s.cnt + (int64_t)blockIdx.x * n;
    int* st = s.start + (int64_t)blockIdx.x * n;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    for (int base = 0; base < n; base += 4 * blockDim.x) {
        const int i0 = base + 4 * threadIdx.x;
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = i0 + u < n ? c[i0 + u] : 0;
        const int tsum = v[0] + v[1] + v[2] + v[3];
        const int incl = wave_incl_scan(tsum);
        if (lane == 63) wsum[wid] = incl;
        __syncthreads();
        int woff = 0, tot = 0;
        for (int w = 0; w < nw; w++) { if (w < wid) woff += wsum[w]; tot += wsum[w]; }
        int e = carry + woff + incl - tsum;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (i0 + u < n && v[u] != 0) st[i0 + u] = e;
            e += v[u];
        }
        __syncthreads();
        if (threadIdx.x == 0) carry += tot;
        __syncthreads();
    }
}

__global__ void k_cl_order(KP P, Bufs B)
{
    const ClSide s = B.cl[blockIdx.y];
    const int64_t total = (int64_t)P.F * s.M;
    for (int64_t it = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; it < total; it += (int64_t)gridDim.x * blockDim.x) {
        const int f = (int)(it / s.M);
        const int m = (int)(it - (int64_t)f * s.M);
        unsigned v = (unsigned)m;
        if (P.K > 0 && blockIdx.y == 0) {
            const int* dp = B.drawn_ptr + (int64_t)f * (P.Mu + 1) + m;
            if (dp[0] < dp[1]) v |= CL_DRAWN;
        }
        s.ord[(int64_t)f * s.M + s.start[((int64_t)f << (3 * s.bits)) + s.key[it]] + s.rank[it]] = (int)v;
    }
}

// atom of row (column) k: the reference atom is the first, so that the loops
// know where its distances are
__device__ __forceinline__ int cl_atom(int k, int iref) { return k == 0 ? iref : (k == iref ? 0 : k); }

// minimum / maximum over groups of `width` consecutive lanes
__device__ __forceinline__ float grp_min(float x, int width)
{
    for (int o = 1; o < width; o <<= 1) x = fminf(x, __shfl_xor(x, o, 64));
    return x;
}
__device__ __forceinline__ float grp_max(float x, int width)
{
    for (int o = 1; o < width; o <<= 1) x = fmaxf(x, __shfl_xor(x, o, 64));
    return x;
}

// The operands, one thread per atom.  blockIdx.z 0: the A tiles, a block per
// super tile, a lane per row; blockIdx.z 1: the B clusters, a wavefront each,
// the lane groups taking the atoms in turn.  blockIdx.y: frame.  Also the boxes
// of tiles, super tiles and clusters, and for the random passes the solute atoms
// and centres (frame of the centre's cell) in the input order.  Padding rows
// and columns are so far away (1e30) that they never pass a test.
template <class T>
__global__ void __launch_bounds__(BLOCK) k_cl_build(KP P, Bufs B, const T* xu, const T* xv)
{
    __shared__ float box[6][CL_SUP], rad[CL_SUP];
    const bool rows = blockIdx.z == 0;
    const int f = blockIdx.y, lane = threadIdx.x & 63, l16 = threadIdx.x & 15;
    const ClSide s = B.cl[rows || P.self_ ? 0 : 1];
    Geo& g = B.geo[f];
    const T* x = (rows || P.self_ ? xu : xv) + (int64_t)f * s.M * s.n * 3;
    const int rpm = P.rpm, mp = 16 / rpm;
    // the tile or cluster, the molecule, its first atom here and the stride
    const int unit = rows ? blockIdx.x * CL_SUP + (threadIdx.x >> 4) : blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6);
    const bool in = unit < (rows ? P.nT : P.nB);
    const int pos = rows ? unit * mp + l16 / rpm : unit * 16 + l16;
    const int a1 = rows ? l16 & (rpm - 1) : lane >> 4;
    const bool on = in && pos < s.M;
    const double* H = g.cell.H;
    double n[3], fr[3], c[3], x0 = 0.0, y0 = 0.0, z0 = 0.0, tx = 0.0, ty = 0.0, tz = 0.0;
    int m = 0, lo3[3], hi3[3];
    for (int k = 0; k < 3; k++) { lo3[k] = 0x7fffffff; hi3[k] = (int)0x80000000; }
    if (on) {
        m = (int)((unsigned)s.ord[(int64_t)f * s.M + pos] & ~CL_DRAWN);
        for (int k = 0; k < 3; k++) c[k] = s.cen[3 * ((int64_t)f * s.M + m) + k];
        load3(x, (int64_t)m * s.n, x0, y0, z0);
        wrap_point(g, c[0], c[1], c[2], fr, n);
        const double sc = ldexp(1.0, g.fix);
        for (int k = 0; k < 3; k++) lo3[k] = hi3[k] = (int)rint(fr[k] * sc);
        tx = H[0] * n[0] + H[3] * n[1] + H[6] * n[2];
        ty = H[1] * n[0] + H[4] * n[1] + H[7] * n[2];
        tz = H[2] * n[0] + H[5] * n[1] + H[8] * n[2];
        if (rows && P.K > 0 && a1 == 0)
            B.ucen[(int64_t)f * P.Mu + m] = mk4((float)(c[0] - tx), (float)(c[1] - ty), (float)(c[2] - tz), __int_as_float(m));
    }
    // fixed-point centre of the tile (cluster): the middle of its molecules' centres
    int ct[3];
    double cx[3];
    for (int k = 0; k < 3; k++) {
        for (int o = 1; o < 16; o <<= 1) {
            lo3[k] = min(lo3[k], __shfl_xor(lo3[k], o, 64));
            hi3[k] = max(hi3[k], __shfl_xor(hi3[k], o, 64));
        }
        ct[k] = lo3[k] <= hi3[k] ? lo3[k] + (hi3[k] - lo3[k]) / 2 : 0;
    }
    const double un = ldexp(1.0, -g.fix);
    for (int k = 0; k < 3; k++) cx[k] = (H[k] * ct[0] + H[3 + k] * ct[1] + H[6 + k] * ct[2]) * un;
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY}, r2 = 0.f;
    if (in)
        for (int q = a1; q < (rows ? rpm : s.n); q += rows ? rpm : 4) {
            const int a = rows && !P.self_ ? q : cl_atom(q, P.iref);
            float e0 = 0.f, e1 = 0.f, e2 = 0.f, w = 1e30f;
            if (on && q < s.n) {
                double xa, ya, za, ox, oy, oz;
                load3(x, (int64_t)m * s.n + a, xa, ya, za);
                cm::minimage(g.cell, xa - x0, ya - y0, za - z0, &ox, &oy, &oz);
                const double px = x0 + ox - tx, py = y0 + oy - ty, pz = z0 + oz - tz;
                e0 = (float)(px - cx[0]); e1 = (float)(py - cx[1]); e2 = (float)(pz - cx[2]);
                w = fmaf(e0, e0, fmaf(e1, e1, e2 * e2));
                lo[0] = fminf(lo[0], e0); lo[1] = fminf(lo[1], e1); lo[2] = fminf(lo[2], e2);
                hi[0] = fmaxf(hi[0], e0); hi[1] = fmaxf(hi[1], e1); hi[2] = fmaxf(hi[2], e2);
                r2 = fmaxf(r2, w);
                if (rows && P.K > 0)
                    B.solw[(int64_t)f * P.Nu + (int64_t)m * s.n + a] = mk4((float)px, (float)py, (float)pz, 0.f);
            }
            float* o = rows ? B.clA + ((int64_t)f * P.nT + unit) * 64 + l16 : B.clB + (((int64_t)f * P.nB + unit) * s.n + q) * 64 + l16;
            o[0] = e0; o[16] = e1; o[32] = e2; o[48] = w;
        }
    const int width = rows ? 16 : 64;
    float l[3], h[3];
    for (int k = 0; k < 3; k++) { l[k] = grp_min(lo[k], width); h[k] = grp_max(hi[k], width); }
    const float r = sqrtf(grp_max(r2, width)) * (1.0f + 1e-6f);
    // (nothing but padding or undefined positions: a box that nothing reaches)
    const bool any = l[0] <= h[0];
    float mid[3], half[3];
    for (int k = 0; k < 3; k++) {
        mid[k] = any ? (float)cx[k] + 0.5f * (l[k] + h[k]) : 0.f;
        half[k] = any ? 0.5f * (h[k] - l[k]) : -1e30f;
    }
    if (in && (lane & (width - 1)) == 0) {
        float4* info = (rows ? B.tinfo + 3 * ((int64_t)f * P.nT + unit) : B.binfo + 3 * ((int64_t)f * P.nB + unit));
        info[0] = fix4(ct[0], ct[1], ct[2], r);
        info[1] = mk4(mid[0], mid[1], mid[2], 0.f);
        info[2] = mk4(half[0], half[1], half[2], 0.f);
    }
    if (!rows || (int)blockIdx.x >= P.nS) return;
    if (l16 == 0) {
        rad[threadIdx.x >> 4] = in ? r : 0.f;
        for (int k = 0; k < 3; k++) {
            box[k][threadIdx.x >> 4] = any ? mid[k] - half[k] : INFINITY;
            box[3 + k][threadIdx.x >> 4] = any ? mid[k] + half[k] : -INFINITY;
        }
    }
    __syncthreads();
    if (threadIdx.x < CL_SUP) {
        float sl[3], sg[3];
        for (int k = 0; k < 3; k++) {
            sl[k] = grp_min(box[k][threadIdx.x], CL_SUP);
            sg[k] = grp_max(box[3 + k][threadIdx.x], CL_SUP);
        }
        // (the maximum rarely grows after the first blocks: a look before the
        // atomic, which the blocks of a frame queue for)
        const float rmax = grp_max(rad[threadIdx.x], CL_SUP);
        if (threadIdx.x == 0) {
            if (rmax > __uint_as_float(__hip_atomic_load(&g.rs_bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
                atomicMax(&g.rs_bits, __float_as_uint(rmax));
            float4* si = B.sinfo + 2 * ((int64_t)f * P.nS + blockIdx.x);
            const bool sany = sl[0] <= sg[0];
            si[0] = sany ? mk4(0.5f * (sl[0] + sg[0]), 0.5f * (sl[1] + sg[1]), 0.5f * (sl[2] + sg[2]), 0.f) : mk4(0.f, 0.f, 0.f, 0.f);
            si[1] = sany ? mk4(0.5f * (sg[0] - sl[0]), 0.5f * (sg[1] - sl[1]), 0.5f * (sg[2] - sl[2]), 0.f) : mk4(-1e30f, -1e30f, -1e30f, 0.f);
        }
    }
}

// Whether a box (mid, half) can come within rc of the wavefront's box (bm, bh)
// under some lattice shift of it by -1, 0 or 1 cells per dimension (all that
// molecules with their centres in the cell can need), and which: bits 0..2,
// 3..5, 6..8 of `sets` for shifts -1, 0, 1 along the three cell vectors.
// Along cell vector k two boxes m cells apart are at least (|f_k + m| - e_k) sp_k
// apart, f the fractions of mid - bm and e those of the half sides.
__device__ __forceinline__ bool cl_reach(const GeoC& g, float rc, float4 mid, float4 half, const float bm[3],
                                         const float bh[3], int& sets)
{
    const float dx = mid.x - bm[0], dy = mid.y - bm[1], dz = mid.z - bm[2];
    const float hx = half.x + bh[0], hy = half.y + bh[1], hz = half.z + bh[2];
    float sum = 0.f;
    bool ok = true;
    sets = 0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const float f = g.Hi32[k] * dx + g.Hi32[3 + k] * dy + g.Hi32[6 + k] * dz;
        const float e = fabsf(g.Hi32[k]) * hx + fabsf(g.Hi32[3 + k]) * hy + fabsf(g.Hi32[6 + k]) * hz;
        float best = INFINITY;
        int set = 0;
#pragma unroll
        for (int m = -1; m <= 1; m++) {
            const float p = fmaxf(fabsf(f + (float)m) - e, 0.f) * (float)g.sp[k];
            set |= p <= rc ? 1 << (m + 1) : 0;
            best = fminf(best, p);
        }
        ok = ok && set != 0;
        sum = fmaf(best, best, sum);
        sets |= set << (3 * k);
    }
    // diagonal cells: the three distances are perpendicular; general ones with
    // a single shift: the boxes' distance along the axes
    if (!ok) return false;
    if (g.ortho) return sum <= rc * rc;
    const int sx = sets & 7, sy = (sets >> 3) & 7, sz = sets >> 6;
    if ((sx & (sx - 1)) | (sy & (sy - 1)) | (sz & (sz - 1))) return true;
    const float m0 = (float)(sx >> 1) - 1.0f, m1 = (float)(sy >> 1) - 1.0f, m2 = (float)(sz >> 1) - 1.0f;
    const float gx = fmaxf(fabsf(dx + (g.H32[0] * m0 + g.H32[3] * m1 + g.H32[6] * m2)) - hx, 0.f);
    const float gy = fmaxf(fabsf(dy + (g.H32[1] * m0 + g.H32[4] * m1 + g.H32[7] * m2)) - hy, 0.f);
    const float gz = fmaxf(fabsf(dz + (g.H32[2] * m0 + g.H32[5] * m1 + g.H32[8] * m2)) - hz, 0.f);
    return fmaf(gx, gx, fmaf(gy, gy, gz * gz)) <= rc * rc;
}

// a value of this lane's row of 16 and of row ^ 1 (O 16) or of row ^ 2 (O 32),
// the lower row's in .x
template <int O>
__device__ __forceinline__ float2 row_pair(float x)
{
    const unsigned u = __float_as_uint(x);
    const auto r = O == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false) : __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return make_float2(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Out of line, with the kernel's arguments read where they are used and the
// histograms by their LDS address (flat atomics took five times as long; glds:
// words before the group histograms, 0: none): the FP64 record of a deferred ...
using CArgs = __attribute__((address_space(4))) const char*;
using LdsU = __attribute__((address_space(3))) unsigned*;
// ... pair (input indices; u < 0: none), by `width` lanes that take its atom pairs
// in turn (sub: this lane's place among them).  One lane a pair walks them all:
// 100 us and more for the few pairs that a wavefront of a small job ends with
// (30 frames of 500 eight-atom molecules in a 60 A box: 164 us, 101 us so)
template <class TU, class TV, bool SELF>
__device__ __attribute__((noinline)) void cl_exact(CArgs k, int f, int u, int v, int sub, int width, LdsU sh_, int glds)
{
    unsigned *const sh = (unsigned*)sh_, *const shg = glds ? sh + glds : nullptr;
    const ClArgs<TU, TV>& A = *(const ClArgs<TU, TV>*)k;
    const KP& P = A.P;
    const TU* x = A.xu + (int64_t)f * P.Nu * 3;
    const TV* y = (SELF ? (const TV*)A.xu : A.xv) + (int64_t)f * P.Nv * 3;
    const int64_t ub = (int64_t)u * P.nu, vb = (int64_t)v * P.nv;
    Rec r1 = rec_zero(), r2 = rec_zero();
    const cm::Cell64& c = A.B.geo[f].cell;
    auto offer = [&](int i, int a, double y0, double y1, double y2) {
        double x0, x1, x2;
        load3(x, ub + i, x0, x1, x2);
        const double d2 = cm::canon_d2(c, x0, x1, x2, y0, y1, y2);
        if (d2 <= P.cut2) {
            const double d = sqrt(d2);
            rec_offer(r1, i, vb + a, d, a == P.iref);
            if (SELF) rec_offer(r2, a, ub + i, d, i == P.iref);
        }
    };
    const int na = u < 0 ? 0 : P.nv;
    double y0, y1, y2;
    if (width <= P.nu) {
        // every lane has some of an atom's pairs
#pragma unroll 1
        for (int a = 0; a < na; a++) {
            load3(y, vb + a, y0, y1, y2);
#pragma unroll 1
            for (int i = sub; i < P.nu; i += width) offer(i, a, y0, y1, y2);
        }
    } else {
#pragma unroll 1
        for (int p = sub; p < na * P.nu; p += width) {
            const int a = p / P.nu;
            load3(y, vb + a, y0, y1, y2);
            offer(p - a * P.nu, a, y0, y1, y2);
        }
    }
    for (int o = 1; o < width; o <<= 1) {
        rec_merge(r1, rec_shfl_xor(r1, o));
        if (SELF) rec_merge(r2, rec_shfl_xor(r2, o));
    }
    if (u < 0 || sub != 0) return;
    const PairCtx<TU, TV, 0> ctx(P, A.B, f, A.xu, A.xv, sh, shg);
    ctx.exact_record(u, v, r1);
    if (SELF) ctx.exact_record(v, u, r2);
}

// ... and the updates of a decided pair where there is more than the plain
// LDS histograms (custom or large groups, dbulk flags)
template <class TU, class TV, bool SELF>
__device__ __attribute__((noinline)) void cl_main(CArgs k, int f, int u, int v, int i, int q, int bin, int bulk, LdsU sh_, int glds)
{
    unsigned *const sh = (unsigned*)sh_, *const shg = glds ? sh + glds : nullptr;
    const ClArgs<TU, TV>& a = *(const ClArgs<TU, TV>*)k;
    const PairCtx<TU, TV, 0> ctx(a.P, a.B, f, a.xu, a.xv, sh, shg);
    if (SELF) ctx.self_main(u, v, i, q, bin, bulk);
    else ctx.cross_main(u, v, i, q, bin, bulk);
}

// Blocks of independent wavefronts that share the LDS histograms; XCD k takes
// the k-th eighth of the (frame, cluster) items in frame-major order, so its L2
// holds one or two frames at a time.
template <class TU, class TV, int RPM, int NVT, bool SELF>
__global__ void __launch_bounds__(NVT > 8 ? 512 : 1024) k_cl_eval(KP P_, Bufs B_, const TU* xu_, const TV* xv_, int S, int Sg_)
{
    constexpr int mp = 16 / RPM, RL = RPM / 4;   // molecules per tile, lane groups per molecule
    constexpr int QB = NVT <= 4 ? 2 : (NVT <= 8 ? 3 : 4);
    // (RPM 1: single atoms on both sides, a row is a molecule and a lane holds four
    // pairs, with nothing to choose between: 30,000 atoms in a 97 A box, 6 frames,
    // 551 us in rows of four, 271 us so; the cell walk 373)
    constexpr bool ONE = RPM == 1;
    constexpr int CBITS = ONE ? 0 : 2 + QB + (RPM == 4 ? 0 : (RPM == 8 ? 1 : 2));   // code: row of the lane, solvent atom, lane group
    constexpr int CMASK = (1 << CBITS) - 1;
    CArgs k0 = (CArgs)__builtin_amdgcn_kernarg_segment_ptr();
    const KP& P = *(const KP*)k0;
    const int gwords = P.glds ? P.nbins * (P.gnu + (SELF ? 0 : P.gnv)) : 0;
    unsigned* const sh = (unsigned*)dyn;
    unsigned* const shg = P.glds ? sh + 2 * P.nbins : nullptr;
    hist_clear(sh, 2 * P.nbins + gwords);
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    // the wavefront's queues: pairs within the cutoff (values, position of the
    // solute molecule, column and doubt), deferred pairs (input indices)
    float* const qv = dyn + ((2 * P.nbins + gwords + 3) & ~3) + wid * CL_WORDS;
    int* const qi = (int*)qv;
    int* const dq = (int*)(qv + 5 * CL_Q);
    float* const tt = qv + 7 * CL_Q;   // centres of the 64 tiles of a turn at their first shift: x, y, z, squared norm
    int qn = 0, dn = 0, fcur = -1, nexact = 0;
    const unsigned long long lt = (1ull << lane) - 1ull;
    const int col = lane & 15, kk = lane >> 4;   // operand component, and the lane group of the results
    const int64_t items = (int64_t)P.F * P.nB * S;
    const int xcd = blockIdx.x & 7, nblk = gridDim.x >> 3;
    const int64_t ihi = items * (xcd + 1) / 8;
    const float pk = ldexpf(1.0f, CBITS - 23);

    auto deferred = [&](int n) {
        wave_sync();
        int w = 1;   // lanes per pair
        CArgs ka = k0;
        asm volatile("" : "+s"(ka));
        const ClArgs<TU, TV>& E = *(const ClArgs<TU, TV>*)ka;
        while (2 * w * n <= 64 && w < E.P.nu * E.P.nv) w *= 2;
        const int e = lane / w, o = 2 * (dn - n + min(e, n - 1));
        cl_exact<TU, TV, SELF>(ka, fcur, e < n ? dq[o] : -1, dq[o + 1], lane & (w - 1), w, (LdsU)sh, shg ? 2 * P.nbins : 0);
        wave_sync();
        dn -= n;
        nexact += n;
    };

    for (int64_t it = items * xcd / 8 + (int64_t)(blockIdx.x >> 3) * nw + wid; it < ihi; it += (int64_t)nblk * nw) {
        CArgs ki = k0;
        asm volatile("" : "+s"(ki));   // fields are read again where they are used (job_args)
        const ClArgs<TU, TV>& A = *(const ClArgs<TU, TV>*)ki;
        // (divisions run on the vector units: their results are scalars again)
        const int64_t fbv = it / S;
        const int f = __builtin_amdgcn_readfirstlane((int)(fbv / A.P.nB));
        const int b = __builtin_amdgcn_readfirstlane((int)(fbv - (int64_t)f * A.P.nB));
        const int64_t fb = (int64_t)f * A.P.nB + b;
        // split items (S > 1): the super tiles in reach go round Sg of them, the
        // tiles of those round S / Sg (Sg from the arguments where it is used: held
        // over the launch it cost 2 % of large ones)
        const int s = (int)(it - fb * S);
        if (f != fcur) {
            while (dn > 0) deferred(min(dn, 64));
            fcur = f;
        }
        const GeoC& g = *(const GeoC*)(A.B.geo + f);
        // the wavefront's cluster: columns (-2 y', |y'|^2) and (-2 y', 1), box
        const int nv = NVT > 4 ? A.P.nv : NVT;
        // (the squares as the products' start, four registers an atom, where
        // there is room, else as the operand's last component: 5 % of the time)
        constexpr bool QUAD = NVT <= 4;
        float Y[NVT], Z[NVT];
        {
            const gptr<const float> cb = (gptr<const float>)(A.B.clB + fb * 64 * A.P.nv);
#pragma unroll
            for (int q = 0; q < NVT; q++) {
                const bool has = q < A.P.nv;
                const float v = has ? cb[q * 64 + lane] : 0.f;
                Y[q] = kk == 3 ? (has ? v : 1e30f) : -2.0f * v;
                Z[q] = kk == 3 ? 1.0f : Y[q];
                if (QUAD) Y[q] = has ? cb[q * 64 + 48 + col] : 1e30f;
            }
        }
        const GeoI3 bc = fix_info(A.B.binfo + 3 * fb);
        const float4 bmid = A.B.binfo[3 * fb + 1], bhalf = A.B.binfo[3 * fb + 2];
        const float bm[3] = {sgpr_f(bmid.x), sgpr_f(bmid.y), sgpr_f(bmid.z)}, bh[3] = {sgpr_f(bhalf.x), sgpr_f(bhalf.y), sgpr_f(bhalf.z)};
        // Guard of the values of pairs within the cutoff (u = 2^-24, S and Y the
        // radii of tile and cluster, t between their centres: |t| <= cutoff + S
        // + Y = W).  s' and y' are rounded by u S and u Y, t by rho u |t| (an
        // exact integer difference): 2 sqrt(3) d times that.  |t - y'|^2, itself
        // at most (d + S)^2: its norms, 3 u each, their sum and four additions to partial
        // sums below Y^2 + 2 Y W + W^2.  The tile: 3 u S^2, the rounding of its
        // columns, 2 u S (d + S), and four additions to sums below (d + 2 S)^2.
        // The low CBITS bits of a value carry its code: below pk of it.
        float Gx, thr;
        {
            const float Sx = __uint_as_float(g.rs_bits), Yx = A.B.binfo[3 * fb].w, cutf = (float)A.P.cutsys + 0.5f;
            const float W = cutf + Sx + Yx, E2 = cutf + 2.0f * Sx;
            const float gx = (0x1p-24f * (4.0f * fmaxf(Yx * (Yx + 2.0f * W), (cutf + Sx) * (cutf + Sx)) + 4.0f * (Yx * Yx + W * W) +
                                          4.0f * E2 * E2 + Sx * (3.0f * Sx + 2.0f * (cutf + Sx)) +
                                          3.5f * cutf * (Sx + Yx + g.rho * W)) + 1e-7f) * (1.0f + 1e-4f);
            Gx = sgpr_f(gx);
            thr = sgpr_f((A.P.c2hi32 + gx) * (1.0f + 1e-6f));
        }
        const float ambx = sgpr_f(2.0f * Gx + (thr + 1.0f) * (pk + 0x1p-21f));

        // counts of up to 64 queued pairs
        auto count = [&](int n) {
            wave_sync();
            const int k = qn - n + lane;
            CArgs kc = k0;
            asm volatile("" : "+s"(kc));
            const ClArgs<TU, TV>& Q = *(const ClArgs<TU, TV>*)kc;
            bool def = false;
            int u = 0, v = 0;
            if (lane < n) {
                const float bv = qv[k], rv = qv[CL_Q + k], ru = SELF ? qv[2 * CL_Q + k] : INFINITY;
                const int info = qi[4 * CL_Q + k];
                const int code = __float_as_int(bv) & CMASK;
                auto decide = [&](float x, int& bin, int& bulk) {
                    const float c = __int_as_float(__float_as_int(x) & ~CMASK) * (1.0f + 0.5f * pk);
                    return decide32(Q.P, Gx + c * (0.5f * pk + 0x1p-21f) + 1e-7f, c, bin, bulk);
                };
                int mbin, mbulk, vbin, ubin = 0, dummy;
                const int dm = decide(bv, mbin, mbulk);
                const int dv = decide(rv, vbin, dummy);
                const int du = SELF ? decide(ru, ubin, dummy) : 1;
                def = dm != 1 && (info >= 256 || dm == 0 || dv == 0 || du == 0);
                const bool plain = shg && !Q.P.gu_ptr && !Q.P.gv_ptr;
                bool drawn = false;
                if (def || !plain || Q.P.K > 0) {
                    const unsigned ou = (unsigned)ldg(Q.B.cl[0].ord + (int64_t)f * Q.P.Mu + qi[3 * CL_Q + k]);
                    const unsigned ov = (unsigned)ldg(Q.B.cl[SELF ? 0 : 1].ord + (int64_t)f * Q.P.Mv + b * 16 + (info & 15));
                    drawn = ((ou | ov) & CL_DRAWN) != 0;
                    u = (int)(ou & ~CL_DRAWN);
                    v = (int)(ov & ~CL_DRAWN);
                }
                if (dm == 2 && !def) {
                    const int row = ONE ? 0 : (code & 3) + (RPM == 4 ? 0 : 4 * (code >> (2 + QB)));
                    const int q = cl_atom((code >> 2) & ((1 << QB) - 1), Q.P.iref), i = SELF ? cl_atom(row, Q.P.iref) : row;
                    const int nb = Q.P.nbins;
                    if (plain && !drawn) {
                        if (mbin < nb) {
                            atomicAdd(&sh[mbin], SELF ? 2u : 1u);
                            atomicAdd(&sh[(2 + i) * nb + mbin], SELF ? 2u : 1u);
                            atomicAdd(&sh[(2 + (SELF ? 0 : Q.P.gnu) + q) * nb + mbin], SELF ? 2u : 1u);
                        }
                    } else cl_main<TU, TV, SELF>(kc, f, u, v, i, q, mbin, mbulk, (LdsU)sh, shg ? 2 * nb : 0);
                    if (dv == 2 && vbin < nb) atomicAdd(&sh[nb + vbin], 1u);
                    if (SELF && du == 2 && ubin < nb) atomicAdd(&sh[nb + ubin], 1u);
                }
            }
            const unsigned long long m = __ballot(def);
            if (def) {
                const int o = 2 * (dn + __popcll(m & lt));
                dq[o] = u;
                dq[o + 1] = v;
            }
            wave_sync();
            qn -= n;
            dn += __popcll(m);
            if (dn >= 64) deferred(64);
        };

        // Tiles in reach: super tiles (a lane each), then the tiles of four of
        // them (a lane each), then one after the other; the next tile's rows
        // are loaded while one is evaluated.  After the last tile the queue is
        // emptied.
        const float rc = (float)A.P.cutsys + 2e-3f + 1e-6f * ((float)g.sp[0] + (float)g.sp[1] + (float)g.sp[2]);
        const gptr<const float> ca = (gptr<const float>)(A.B.clA + (int64_t)f * A.P.nT * 64);
        const int nS = A.P.nS;
        int turn = 0, sturn = 0;   // tiles, super tiles in reach so far (split items)
        int sb = -64;
        unsigned long long smask = 0, tm = 0;
        int tile = 0, sets = 0, tn = -1;
        float an = 0.f;
        // a lane's tile: its centre from the cluster's in fixed point; of the next
        // tile that and its operand component
        int ci[3] = {0, 0, 0}, sn = 0, nx[3] = {0, 0, 0};
        float nt = 0.f;
        bool more = true;
        for (;;) {
            const float a = an;
            const int t = tn, st = sn, dx = nx[0], dy = nx[1], dz = nx[2];
            float nt0 = nt;
            tn = -1;
            while (tm == 0 && more) {
                CArgs kr = k0;
                asm volatile("" : "+s"(kr));
                const ClArgs<TU, TV>& R = *(const ClArgs<TU, TV>*)kr;
                const GeoC& gr = *(const GeoC*)(R.B.geo + f);
                if (smask == 0) {
                    sb += 64;
                    if (sb >= nS) { more = false; break; }
                    bool in = false;
                    if (sb + lane < nS) {
                        const float4* si = R.B.sinfo + 2 * ((int64_t)f * nS + sb + lane);
                        in = cl_reach(gr, rc, si[0], si[1], bm, bh, sets);
                    }
                    smask = __ballot(in);
                    if (S > 1 && R.Sg > 1) {
                        const int rank = sturn + __popcll(smask & lt);
                        sturn = __builtin_amdgcn_readfirstlane((sturn + __popcll(smask)) % R.Sg);
                        smask = __ballot(in && rank % R.Sg == s % R.Sg);
                    }
                    continue;
                }
                int mine = -1;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int bit = smask ? __ffsll((long long)smask) - 1 : -1;
                    if (smask) smask &= smask - 1ull;
                    mine = kk == j ? bit : mine;
                }
                tile = (sb + mine) * CL_SUP + col;
                bool ok = false;
                sets = 0;
                // Self mode: a cluster's own molecules pair once; two blocks of 16
                // molecules meet in the cluster that the parity of their sum
                // names, which shares the work evenly (upper ones alone leave
                // the first clusters twice the mean and the last ones nothing).
                const int ub = tile * mp / 16;
                if (mine >= 0 && tile < R.P.nT && (!SELF || ub == b || ((ub + b) & 1) == (ub > b ? 1 : 0))) {
                    const float4* ti = R.B.tinfo + 3 * ((int64_t)f * R.P.nT + tile);
                    ok = cl_reach(gr, rc, ti[1], ti[2], bm, bh, sets);
                    const float4 t0 = ti[0];
                    ci[0] = __float_as_int(t0.x) - bc.x; ci[1] = __float_as_int(t0.y) - bc.y; ci[2] = __float_as_int(t0.z) - bc.z;
                    const int one = 1 << gr.fix;
                    float tx, ty, tz;
                    fix_cart(gr, ci[0] + (__builtin_ctz(sets | 8) - 1) * one, ci[1] + (__builtin_ctz((sets >> 3) | 8) - 1) * one,
                             ci[2] + (__builtin_ctz((sets >> 6) | 8) - 1) * one, tx, ty, tz);
                    *(float4*)&tt[4 * lane] = mk4(tx, ty, tz, fmaf(tx, tx, fmaf(ty, ty, tz * tz)));
                }
                wave_sync();
                tm = __ballot(ok);
                if (S > 1) {
                    const int rank = turn + __popcll(tm & lt), St = S / R.Sg;
                    turn = __builtin_amdgcn_readfirstlane((turn + __popcll(tm)) % St);
                    tm = __ballot(ok && rank % St == s / R.Sg);
                }
            }
            if (tm) {
                const int bit = __ffsll((long long)tm) - 1;
                tm &= tm - 1ull;
                tn = __builtin_amdgcn_readlane(tile, bit);
                sn = __builtin_amdgcn_readlane(sets, bit);
#pragma unroll
                for (int k = 0; k < 3; k++) nx[k] = __builtin_amdgcn_readlane(ci[k], bit);
                nt = tt[4 * bit + kk];
                an = ca[(int64_t)tn * 64 + lane];
            }
            if (t >= 0) {
                float bb = INFINITY, ms = INFINITY, rv = INFINITY, ru = INFINITY;
                f4m one = {INFINITY, INFINITY, INFINITY, INFINITY};   // ONE: the lane's pairs
                int xs = st & 7, ys = (st >> 3) & 7, zs = st >> 6;
                for (;;) {
                    const float at = kk == 3 ? 1.0f : nt0, ct = kk == 3 ? nt0 : 0.f, bt = kk == 3 ? 0.f : 2.0f * nt0;
#pragma unroll
                    for (int q = 0; q < NVT; q++) {
                        if (NVT > 4 && (q & 1) == 0 && q >= nv) break;   // (by twos: independent chains)
                        // |t - y'|^2 in every row, then the distances
                        const f4m c = QUAD ? __builtin_amdgcn_mfma_f32_16x16x4f32(nt0, Z[q], f4m{Y[q], Y[q], Y[q], Y[q]}, 0, 0, 0)
                                           : __builtin_amdgcn_mfma_f32_16x16x4f32(at, Y[q] + ct, f4m{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        f4m d = __builtin_amdgcn_mfma_f32_16x16x4f32(a, Z[q] + bt, c, 0, 0, 0);
                        if constexpr (ONE) {
#pragma unroll
                            for (int r = 0; r < 4; r++) one[r] = fminf(one[r], d[r]);
                            continue;
                        }
#pragma unroll
                        for (int r = 0; r < 4; r++) d[r] = __int_as_float((__float_as_int(d[r]) & ~CMASK) | (r | (q << 2)));
                        min2_4(bb, ms, d);
                        if (q == 0) {
                            rv = fminf(fminf(rv, d[0]), d[1]);
                            rv = fminf(fminf(rv, d[2]), d[3]);
                        }
                        if (SELF) ru = fminf(ru, d[0]);
                    }
                    // further shifts in reach (boxes that two images of a tile reach)
                    xs &= xs - 1;
                    if (!xs) { xs = st & 7; ys &= ys - 1; }
                    if (!ys) { ys = (st >> 3) & 7; zs &= zs - 1; }
                    if (!zs) break;
                    float tx, ty, tz;
                    fix_cart(g, dx + (__builtin_ctz(xs) - 1) * (1 << g.fix), dy + (__builtin_ctz(ys) - 1) * (1 << g.fix),
                             dz + (__builtin_ctz(zs) - 1) * (1 << g.fix), tx, ty, tz);
                    nt0 = kk == 0 ? tx : (kk == 1 ? ty : (kk == 2 ? tz : fmaf(tx, tx, fmaf(ty, ty, tz * tz))));
                }
                if constexpr (ONE) {
                    // (two images of a molecule within reach: the nearer one)
#pragma unroll 1
                    for (int r = 0; r < 4; r++) {
                        const float x = one[0];
                        one = f4m{one[1], one[2], one[3], INFINITY};
                        unsigned long long m = __ballot(x <= thr);
                        if (SELF && t == b) m &= __ballot(4 * kk + r > col);
                        if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                            const int k = qn + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
                            qv[k] = x; qv[CL_Q + k] = x;
                            if (SELF) qv[2 * CL_Q + k] = x;
                            qi[3 * CL_Q + k] = t * mp + 4 * kk + r;
                            qi[4 * CL_Q + k] = col;
                        }
                        qn += __popcll(m);
                        if (r < 3 && qn >= 64) count(64);
                    }
                }
                // lane groups holding the other rows of the molecule
                if constexpr (RPM > 4) {
                    bb = __int_as_float(__float_as_int(bb) | ((kk & (RL - 1)) << (2 + QB)));
                    if (SELF) ru = (kk & (RL - 1)) == 0 ? ru : INFINITY;
                    auto merge = [&](auto pair) {
                        const float2 b2 = pair(bb), s2 = pair(ms), v2 = pair(rv);
                        ms = fminf(fminf(fmaxf(b2.x, b2.y), s2.x), s2.y);
                        bb = fminf(b2.x, b2.y);
                        rv = fminf(v2.x, v2.y);
                        if (SELF) {
                            const float2 u2 = pair(ru);
                            ru = fminf(u2.x, u2.y);
                        }
                    };
                    merge([](float x) { return row_pair<16>(x); });
                    if constexpr (RPM > 8) merge([](float x) { return row_pair<32>(x); });
                }
                if constexpr (!ONE) {
                    const int up = t * mp + (RPM == 4 ? kk : (RPM == 8 ? kk >> 1 : 0));
                    unsigned long long m = __ballot((RPM == 4 || (kk & (RL - 1)) == 0) && bb <= thr);
                    if (SELF && t * mp / 16 == b) m &= __ballot((up & 15) > col);
                    const bool hit = __builtin_amdgcn_inverse_ballot_w64(m);
                    if (hit) {
                        const int k = qn + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
                        qv[k] = bb; qv[CL_Q + k] = rv;
                        if (SELF) qv[2 * CL_Q + k] = ru;
                        qi[3 * CL_Q + k] = up;
                        qi[4 * CL_Q + k] = col | (ms - bb > ambx ? 0 : 256);
                    }
                    qn += __popcll(m);
                }
            }
            const bool last = tn < 0 && t < 0 && !more;
            if (qn >= 64 || last) count(min(qn, 64));
            if (last) break;
        }
    }
    while (dn > 0) deferred(min(dn, 64));
    // (one atomic a block: on a single address they take about 10 ns each)
    if (lane == 0) qi[0] = nexact;
    __syncthreads();
    if (threadIdx.x == 0) {
        ull n = 0;
        for (int w = 0; w < nw; w++) n += (ull)qi[w * CL_WORDS];
        if (n) atomicAdd(&B_.stats[0], SELF ? 2 * n : n);
    }
    hist_flush(sh, P.nbins, B_.cnt_md, B_.cnt_rdf);
    if (shg) groups_flush(P, shg, B_.cnt_gu, B_.cnt_gv);
}

// Ranges of memory, each filled with copies of its own word, all in one launch:
// nine of a small call's thirty launches were fills, some 4 us each.  (A kernel,
// not hipMemsetAsync: memset nodes captured in HIP graphs have given wrong
// results on replays here, and a caller may capture these launches.)
struct FillList {
    static constexpr int MAX = 6;   // (the longest list has five)
    int n = 0;
    unsigned char* p[MAX];   // 16-byte aligned: every buffer here starts on a 256-byte boundary
    int64_t bytes[MAX];
    unsigned word[MAX];
    void add(void* q, size_t b, unsigned w = 0)
    {
        if (!b) return;
        p[n] = (unsigned char*)q;
        bytes[n] = (int64_t)b;
        word[n++] = w;
    }
};
__global__ void k_fill(FillList L)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    for (int r = 0; r < L.n; r++) {
        uint4* p = (uint4*)L.p[r];
        const unsigned w = L.word[r];
        const int64_t n16 = L.bytes[r] >> 4;
        for (int64_t k = t; k < n16; k += stride) p[k] = make_uint4(w, w, w, w);
        if (t < (L.bytes[r] & 15)) L.p[r][16 * n16 + t] = (unsigned char)(w >> (8 * (t & 3)));
    }
}

// verification records of molecules no chunk evaluates: not within the
// cutoff (zero(MinimumDistance), src/minimum_distances.jl:21-28)
__global__ void k_vrec_init(VRec* p, int64_t n)
{
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        VRec o;
        o.within = 0; o.i = -1; o.j = -1; o.d = INFINITY; o.ref = 0; o.pad = 0; o.dref = INFINITY;
        p[k] = o;
    }
}

// integer hits -> FP64 accumulators (assign: the first run of the job, every
// entry written, so the accumulators need not hold zeros)
__global__ void k_flush(ull* cnt, double* acc, ull* hits, int64_t n, int64_t nhist, int64_t half_lo, int64_t half_hi,
                        double w, int assign)
{
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        ull c = cnt[k];
        double mult = (k >= half_lo && k < half_hi) ? w / 2 : w;
        if (assign) {
            acc[k] = (double)c * mult;
        } else {
            if (!c) continue;
            acc[k] += (double)c * mult;
        }
        if (k < nhist) hits[k] += c;
        cnt[k] = 0ull;
    }
}

// Read-back of a job whose frames all had one weight: the md/rdf hits are
// added to the cumulative ones (read back as 64-bit words); each group count
// goes out as a 16-bit word, and the counts that do not fit (0xffff and up)
// are listed as (entry, count) in ov, at most ovcap of them (over[1] counts
// them all).  over[0] is set when a count exceeds limit (at most 2^32 - 1).
// The counts stay in cnt for the FP64 path.
__global__ void k_pack16(const ull* cnt, uint16_t* out, ull* hits, int64_t n, int64_t nhist, ull limit, ull* over,
                         ulonglong2* ov, int64_t ovcap)
{
    bool big = false;
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
        const ull c = cnt[k];
        big |= c > limit;
        if (k < nhist) {
            hits[k] += c;
            continue;
        }
        out[k - nhist] = (uint16_t)(c < 0xffffull ? c : 0xffffull);
        if (c >= 0xffffull) {
            const ull slot = atomicAdd(&over[1], 1ull);
            if (slot < (ull)ovcap) ov[slot] = make_ulonglong2((ull)k, c);
        }
    }
    if (big) atomicOr(&over[0], 1ull);
}

// ---------------------------------------------------------------------------
// many jobs per launch (cm_jobs_submit_device): one round runs one batch of
// frames of every job, and each stage of the single-solute path is one launch
// over all of them.  A device table holds each job's parameters and buffers
// and, per stage, how many blocks of that stage's single-job grid the job has;
// every block of a stage launch walks the concatenated block lists (a block
// index maps to a job by a search over the prefix of the counts), so one
// launch does exactly the work of the jobs' own launches.  The launches read
// nothing but the table's address: a round is a table upload plus the same
// launch sequence, which is captured once in a HIP graph and replayed.
// ---------------------------------------------------------------------------
constexpr int MS_MAX = 128;   // jobs per round
enum MStage {
    MS_ZERO, MS_RADII, MS_WRAP, MS_SCAN_CELLS, MS_SCATTER, MS_NEAR, MS_DFIELD, MS_PREP, MS_SCAN_SUMS0,
    MS_SCAN_ROWS0, MS_MOL_SCATTER0, MS_FILL, MS_CHUNK0, MS_BULK_INIT, MS_BULK_COMPACT, MS_PLACE_KEYS, MS_SCAN_SUMSK,
    MS_SCAN_ROWSK, MS_MOL_SCATTERK, MS_PLACE_NEAR, MS_CHUNKK, MS_RESOLVE0, MS_RESOLVEK, MS_N
};

struct SysDev {
    KP P;
    Bufs B;
    const void* xu;          // device coordinates of the round's frames
    const void* xv;
    uint4* zp[3];            // buffers cleared at the start of the round (cell counts, near flags, key counts)
    int64_t z16[3];          // their sizes in 16-byte words
    int nbx[MS_N];           // x extent (blocks) of each stage's grid for this job; y = blocks / nbx
};

struct MultiTab {
    int nsys;
    int pad;
    int base[MS_N][MS_MAX + 1];   // per stage: prefix over the jobs of their block counts
    SysDev sys[MS_MAX];
};

// Runs fn(job, bx, nbx, by, nby) for every (job, block) of stage ST, the
// block indices of the launch striding over the concatenated lists.  SYNC:
// the stage's body uses shared memory, so the block synchronises between two
// of its virtual blocks.
template <int ST, bool SYNC, class Fn>
__device__ __forceinline__ void multi_blocks(const MultiTab* __restrict__ MT, Fn fn)
{
    // the stage's prefix row in LDS; a block's virtual blocks increase, so
    // its job index only moves forward
    __shared__ int base[MS_MAX + 1];
    const int n = MT->nsys;
    for (int k = threadIdx.x; k <= n; k += blockDim.x) base[k] = MT->base[ST][k];
    __syncthreads();
    // values read from LDS are the same in every lane; made uniform, the
    // job's parameters below are scalar loads, as kernel arguments would be
    const int total = __builtin_amdgcn_readfirstlane(base[n]);
    int lo = 0;
    for (int vb = blockIdx.x; vb < total; vb += gridDim.x) {
        while (base[lo + 1] <= vb) lo++;
        lo = __builtin_amdgcn_readfirstlane(lo);
        const int b0 = __builtin_amdgcn_readfirstlane(base[lo]), b1 = __builtin_amdgcn_readfirstlane(base[lo + 1]);
        const SysDev& S = MT->sys[lo];
        const int local = vb - b0;
        const int nbx = S.nbx[ST];
        const int nby = (b1 - b0) / nbx;
        fn(S, local - (local / nbx) * nbx, nbx, local / nbx, nby);
        if (SYNC) __syncthreads();
    }
}

__global__ void km_zero(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_ZERO, false>(MT, [&](const SysDev& S, int bx, int nbx, int, int) {
        const int64_t n0 = S.z16[0], n1 = S.z16[1], tot = n0 + n1 + S.z16[2];
        for (int64_t k = bx * (int64_t)blockDim.x + threadIdx.x; k < tot; k += (int64_t)nbx * blockDim.x) {
            uint4* q = k < n0 ? S.zp[0] + k : (k < n0 + n1 ? S.zp[1] + (k - n0) : S.zp[2] + (k - n0 - n1));
            *q = make_uint4(0u, 0u, 0u, 0u);
        }
    });
}

template <class T>
__global__ void __launch_bounds__(BLOCK) km_radii(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_RADII, true>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_radii<T>(S.P, S.B, (const T*)S.xu, (const T*)S.xv, 0, bx, nbx, by, nby);
    });
}

template <class T>
__global__ void km_wrap_atoms(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_WRAP, false>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_wrap_atoms<T>(S.P, S.B, (const T*)S.xu, bx, nbx, by, nby);
    });
}

__global__ void __launch_bounds__(1024) km_scan_cells(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_SCAN_CELLS, true>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_scan_cells(S.P, S.B, bx, nbx, by, nby);
    });
}

__global__ void km_scatter(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_SCATTER, false>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_scatter(S.P, S.B, S.B.nitems, bx, nbx, by, nby);
    });
}

__global__ void km_near_mark(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_NEAR, true>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_near_mark(S.P, S.B, bx, nbx, by, nby);
    });
}

__global__ void km_dfield(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_DFIELD, false>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_dfield(S.P, S.B, bx, nbx, by, nby);
    });
}

template <class T>
__global__ void km_prep_solvent_tiles(const MultiTab* __restrict__ MT)
{
    __shared__ unsigned tab[48];
    hilbert_load(tab);
    multi_blocks<MS_PREP, false>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_prep_solvent_tiles<T>(S.P, S.B, (const T*)S.xv, tab, bx, nbx, by, nby);
    });
}

template <bool RANDOM>
__global__ void __launch_bounds__(1024) km_scan_rows(const MultiTab* __restrict__ MT)
{
    multi_blocks<RANDOM ? MS_SCAN_ROWSK : MS_SCAN_ROWS0, true>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_scan_rows(S.P, S.B, RANDOM ? 1 : 0, bx, nbx, by, nby);
    });
}

template <bool RANDOM>
__global__ void __launch_bounds__(1024) km_scan_sums(const MultiTab* __restrict__ MT)
{
    multi_blocks<RANDOM ? MS_SCAN_SUMSK : MS_SCAN_SUMS0, true>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_scan_sums(S.P, S.B, RANDOM ? 1 : 0, bx, nbx, by, nby);
    });
}

template <bool RANDOM>
__global__ void km_mol_scatter(const MultiTab* __restrict__ MT)
{
    multi_blocks<RANDOM ? MS_MOL_SCATTERK : MS_MOL_SCATTER0, false>(MT, [&](const SysDev& S, int bx, int nbx, int by,
                                                                            int nby) {
        b_mol_scatter(S.P, S.B, RANDOM ? 1 : 0, bx, nbx, by, nby);
    });
}

template <class T>
__global__ void km_fill_real(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_FILL, false>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_fill_real<T>(S.P, S.B, (const T*)S.xv, bx, nbx, by, nby);
    });
}

template <bool RANDOM>
__global__ void __launch_bounds__(1024) km_chunk_table(const MultiTab* __restrict__ MT)
{
    multi_blocks<RANDOM ? MS_CHUNKK : MS_CHUNK0, true>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_chunk_table<true>(S.P, S.B, RANDOM ? 1 : 0, bx, nbx, by, nby);
    });
}

__global__ void km_bulk_init(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_BULK_INIT, false>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_bulk_init(S.P, S.B, bx, nbx, by, nby);
    });
}

__global__ void __launch_bounds__(1024) km_bulk_compact(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_BULK_COMPACT, true>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_bulk_compact(S.P, S.B, bx, nbx, by, nby);
    });
}

__global__ void km_place_keys(const MultiTab* __restrict__ MT)
{
    __shared__ unsigned tab[48];
    hilbert_load(tab);
    multi_blocks<MS_PLACE_KEYS, false>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_place_keys(S.P, S.B, tab, bx, nbx, by, nby);
    });
}

template <class T>
__global__ void km_place_near(const MultiTab* __restrict__ MT)
{
    multi_blocks<MS_PLACE_NEAR, false>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_place_near<T>(S.P, S.B, (const T*)S.xv, bx, nbx, by, nby);
    });
}

// The chunks of every job of a round in tickets of about `per` chunks of one
// job, taken by blocks from the counter ctr (zero at the start of the launch):
// a ticket's chunks lie at a stride over its job, so the tickets of a job cost
// about the same.  The LDS histograms belong to one job: a block flushes them
// when its next ticket is another job's.  body(job, hist, chunk) runs per
// wavefront; tab: words of the chunk tables' place in LDS, 3 (MS_MAX + 1).
template <bool RANDOM, class Fn>
__device__ __forceinline__ void multi_tickets(const MultiTab* __restrict__ MT, int* ctr, Fn body)
{
    __shared__ int nch[MS_MAX], tk[MS_MAX + 1], s_t;
    const int n = MT->nsys;
    for (int j = threadIdx.x; j < n; j += blockDim.x) {
        const KP& Pj = MT->sys[j].P;
        nch[j] = (RANDOM && Pj.K == 0) ? 0 : MT->sys[j].B.chunk_base[Pj.F * (RANDOM ? Pj.NG : 1)];
    }
    __syncthreads();
    const int nw = blockDim.x >> 6;
    if (threadIdx.x == 0) {
        int64_t total = 0;
        for (int j = 0; j < n; j++) total += nch[j];
        const int per = (int)max((int64_t)nw, min((int64_t)16 * nw, total / ((int64_t)gridDim.x * 8)));
        int acc = 0;
        for (int j = 0; j < n; j++) {
            tk[j] = acc;
            acc += (nch[j] + per - 1) / per;
        }
        tk[n] = acc;
    }
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int cur = -1;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_t = atomicAdd(ctr, 1);
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(s_t);
        if (t >= tk[n]) break;
        int lo = 0, hi = n;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (tk[mid] <= t) lo = mid; else hi = mid;
        }
        lo = __builtin_amdgcn_readfirstlane(lo);
        if (lo != cur) {
            if (cur >= 0) ev_hist_flush<RANDOM>(MT->sys[cur].P, MT->sys[cur].B);
            __syncthreads();
            ev_hist_clear(MT->sys[lo].P);
            __syncthreads();
            cur = lo;
        }
        const int nt = tk[lo + 1] - tk[lo], nc = nch[lo];
        for (int ch = t - tk[lo] + wid * nt; ch < nc; ch += nw * nt) body(MT->sys[lo], ch);
    }
    if (cur >= 0) ev_hist_flush<RANDOM>(MT->sys[cur].P, MT->sys[cur].B);
}

template <class TU, class TV, bool RANDOM, int G, int TQ>
__global__ void __launch_bounds__(1024) km_eval_tiles(const MultiTab* __restrict__ MT, int* ctr)
{
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    multi_tickets<RANDOM>(MT, ctr, [&](const SysDev& S, int ch) {
        const EvHist hist(S.P);
        auto base = [&](int k) { return ldg(S.B.chunk_base + k); };
        const ChunkAt at(S.P, S.B, RANDOM, ch, base);
        eval_chunk<TU, TV, RANDOM, G, TQ, false>(S.P, S.B, (const TU*)S.xu, (const TV*)S.xv, ch, at,
                                                ((EvHist::words(S.P) + 3) & ~3) + wid * eval_wave_words(G, TQ), hist);
    });
}

template <class TU, class TV, bool RANDOM>
__global__ void __launch_bounds__(BLOCK, 3) km_resolve(const MultiTab* __restrict__ MT)
{
    multi_blocks<RANDOM ? MS_RESOLVEK : MS_RESOLVE0, true>(MT, [&](const SysDev& S, int bx, int nbx, int by, int nby) {
        b_resolve<TU, TV, RANDOM, false>(S.P, S.B, (const TU*)S.xu, (const TV*)S.xv, bx, nbx, by, nby);
    });
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
thread_local std::string g_err;

int fail(int code, const std::string& msg)
{
    g_err = msg;
    return code;
}

#define HIPCHK(x)                                                                                  \
    do {                                                                                           \
        hipError_t e_ = (x);                                                                       \
        if (e_ != hipSuccess) return fail(CM_EHIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

// blocks per frame of k_near_mark: every lane an item while that is few blocks
// (each clears and writes out its bitmap), then as many as there are atoms for
int near_blocks(int nu)
{
    const int all = (int)(((int64_t)nu * near_lanes(nu) + BLOCK - 1) / BLOCK);
    return std::max(1, std::min(all, std::max(4, (nu + BLOCK - 1) / BLOCK)));
}

// x: blocks over n molecules or slots; y: one per (frame, pass) pair, up to
// the grid limit (the kernels stride over y beyond it)
dim3 grid_slots(int n, int pairs)
{
    return dim3((unsigned)std::max(1, (n + BLOCK - 1) / BLOCK), (unsigned)std::max(1, std::min(pairs, 65535)));
}

int grid_for(int64_t n)
{
    int64_t b = (n + BLOCK - 1) / BLOCK;
    if (b < 1) b = 1;
    if (b > 4096) b = 4096;
    return (int)b;
}

// one launch of k_fill over the ranges of L on stream s, a lane per 16 bytes of
// the longest up to 2,048 blocks
int fill_async(const FillList& L, hipStream_t s)
{
    if (!L.n) return CM_OK;
    int64_t n16 = 1;
    for (int r = 0; r < L.n; r++) n16 = std::max(n16, L.bytes[r] >> 4);
    hipLaunchKernelGGL(k_fill, dim3((unsigned)std::min<int64_t>((n16 + BLOCK - 1) / BLOCK, 2048)), dim3(BLOCK), 0, s, L);
    HIPCHK(hipGetLastError());
    return CM_OK;
}

struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
};

// Memory released by finished jobs, kept for the next ones (a process that
// runs one mddf call after another would otherwise pay hipMalloc/hipFree,
// which synchronise the device, for about 1 GB of batch scratch and tens of
// MB of page-locked read-back buffers per call).  Blocks are reused for
// requests of at least half their size; beyond a cap the largest are
// released.  Heap singletons: never destroyed, so nothing runs at exit.
struct BlockCache {
    std::mutex m;
    std::multimap<size_t, std::pair<int, void*>> blocks;   // bytes -> (device, pointer)
    size_t total = 0;
};

BlockCache& dev_cache()
{
    static BlockCache* c = new BlockCache;
    return *c;
}

BlockCache& pin_cache()
{
    static BlockCache* c = new BlockCache;
    return *c;
}

constexpr size_t DEV_CACHE_MAX = (size_t)48 << 30;
constexpr size_t PIN_CACHE_MAX = (size_t)4 << 30;

void* cache_take(BlockCache& c, size_t bytes, int dev, size_t* got)
{
    std::lock_guard<std::mutex> lk(c.m);
    for (auto it = c.blocks.lower_bound(bytes); it != c.blocks.end() && it->first <= 2 * bytes; ++it) {
        if (it->second.first != dev) continue;
        void* p = it->second.second;
        *got = it->first;
        c.total -= it->first;
        c.blocks.erase(it);
        return p;
    }
    return nullptr;
}

// returns a block; blocks beyond the cap (largest first) come back to be freed
std::vector<std::pair<int, void*>> cache_put(BlockCache& c, void* p, size_t bytes, int dev, size_t cap)
{
    std::vector<std::pair<int, void*>> out;
    std::lock_guard<std::mutex> lk(c.m);
    c.blocks.emplace(bytes, std::make_pair(dev, p));
    c.total += bytes;
    while (c.total > cap && !c.blocks.empty()) {
        auto it = std::prev(c.blocks.end());
        c.total -= it->first;
        out.push_back(it->second);
        c.blocks.erase(it);
    }
    return out;
}

std::vector<std::pair<int, void*>> cache_drain(BlockCache& c)
{
    std::lock_guard<std::mutex> lk(c.m);
    std::vector<std::pair<int, void*>> out;
    for (auto& kv : c.blocks) out.push_back(kv.second);
    c.blocks.clear();
    c.total = 0;
    return out;
}

int current_device()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) dev = 0;
    return dev;
}

// device block of at least `bytes`: a cached one, else hipMalloc (after
// releasing the cache when the device is full)
int dev_take(DevBuf& b, size_t bytes)
{
    const int dev = current_device();
    size_t got = 0;
    if (void* p = cache_take(dev_cache(), bytes, dev, &got)) {
        b.p = p;
        b.bytes = got;
        return CM_OK;
    }
    hipError_t e = hipMalloc(&b.p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        for (auto& blk : cache_drain(dev_cache())) (void)hipFree(blk.second);
        e = hipMalloc(&b.p, bytes);
    }
    if (e != hipSuccess) {
        b.p = nullptr;
        return fail(CM_ENOMEM, std::string("hipMalloc failed for ") + std::to_string(bytes) + " bytes");
    }
    b.bytes = bytes;
    return CM_OK;
}

// a block no stream uses any more goes back to the cache
void dev_put(DevBuf& b)
{
    if (!b.p) return;
    for (auto& blk : cache_put(dev_cache(), b.p, b.bytes, current_device(), DEV_CACHE_MAX)) (void)hipFree(blk.second);
    b.p = nullptr;
    b.bytes = 0;
}

struct PinBuf {
    void* p = nullptr;
    size_t bytes = 0;
};

int pin_take(PinBuf& b, size_t bytes)
{
    size_t got = 0;
    if (void* p = cache_take(pin_cache(), bytes, 0, &got)) {
        b.p = p;
        b.bytes = got;
        return CM_OK;
    }
    if (hipHostMalloc(&b.p, bytes, hipHostMallocDefault) != hipSuccess) {
        b.p = nullptr;
        return fail(CM_ENOMEM, std::string("hipHostMalloc failed for ") + std::to_string(bytes) + " bytes");
    }
    b.bytes = bytes;
    return CM_OK;
}

void pin_put(PinBuf& b)
{
    if (!b.p) return;
    for (auto& blk : cache_put(pin_cache(), b.p, b.bytes, 0, PIN_CACHE_MAX)) (void)hipHostFree(blk.second);
    b.p = nullptr;
    b.bytes = 0;
}

// Streams of destroyed jobs, kept per device for the next ones: a process
// that runs one mddf call after another would otherwise create and destroy a
// stream per call.  A stream comes back idle (cm_job_destroy waits for it).
struct StreamPool {
    std::mutex m;
    std::vector<std::pair<int, hipStream_t>> s;   // (device, stream)
};

StreamPool& stream_pool()
{
    static StreamPool* p = new StreamPool;
    return *p;
}

constexpr size_t STREAM_POOL_MAX = 64;

int stream_take(hipStream_t* out)
{
    const int dev = current_device();
    {
        StreamPool& p = stream_pool();
        std::lock_guard<std::mutex> lk(p.m);
        for (size_t k = p.s.size(); k-- > 0;)
            if (p.s[k].first == dev) {
                *out = p.s[k].second;
                p.s.erase(p.s.begin() + k);
                return CM_OK;
            }
    }
    if (hipStreamCreateWithFlags(out, hipStreamNonBlocking) != hipSuccess) {
        *out = nullptr;
        return fail(CM_EHIP, "hipStreamCreate failed");
    }
    return CM_OK;
}

void stream_put(hipStream_t st)
{
    if (!st) return;
    int dev = 0;
    if (hipStreamGetDevice(st, &dev) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipStreamDestroy(st);
        return;
    }
    StreamPool& p = stream_pool();
    {
        std::lock_guard<std::mutex> lk(p.m);
        if (p.s.size() < STREAM_POOL_MAX) {
            p.s.emplace_back(dev, st);
            return;
        }
    }
    (void)hipStreamDestroy(st);
}

// host memory the runtime knows as page-locked (hipHostMalloc'd or registered)
bool page_locked(const void* p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();   // pageable memory is unknown to the runtime
        return false;
    }
    return a.type == hipMemoryTypeHost;
}

void plane_spacings(const double* H, double sp[3])
{
    double V = std::fabs(cm::cell_volume(H));
    for (int k = 0; k < 3; k++) {
        const double *p = H + 3 * ((k + 1) % 3), *q = H + 3 * ((k + 2) % 3);
        double x = p[1] * q[2] - p[2] * q[1], y = p[2] * q[0] - p[0] * q[2], z = p[0] * q[1] - p[1] * q[0];
        sp[k] = V / std::sqrt(x * x + y * y + z * z);
    }
}

}  // namespace

struct cm_job {
    cm_job_desc d;
    KP kp;
    bool atoms_family = true;
    hipStream_t stream = nullptr;
    int64_t Nu = 0, Nv = 0;
    int K = 0, kb = 0;
    // accumulators: [md | md_r | rdf | rdf_r | gu | gv | gu_r | gv_r]
    int64_t acc_len = 0;
    DevBuf cnt, acc, hits, stats;
    double pending_w = 0.0;
    bool pending = false;
    int64_t flushes = 0;   // weight runs already added to the FP64 accumulators
    double volume_total = 0.0;
    DevBuf gmap;   // group maps
    // batch buffers
    DevBuf geo, cells_cnt, cells_start, tmp4, tmpcell, sorted, solw, ucen, vw, vcell, vcen;
    DevBuf P, vw_r, vcen_r, bflag, blist, nbulk, uk, drawn_ptr, drawn_idx;
    DevBuf clmem;             // molecule pairs on the matrix cores: one block for all their buffers
    DevBuf near, mkey, mrank, mcnt, mstart, msum, msorted, nnear, chunk_base;
    DevBuf xin_u, xin_v;
    double cell_frac = 0.5;   // tiles family: fine cell side as a fraction of the cutoff
    int tile_c = 4;           // tiles family: 64 / (molecules per chunk of the real pass; atoms unless 3 per molecule): 1, 2, 4 or 8
    bool tuned_c = false;     // tile_c was set (cm_job_set_tuning): chunks keep that size
    int eval_grid = 0;        // tiles family: workgroups of the persistent evaluation kernel (0: fill the device)
    int cus = 256;            // compute units of the device
    int lds_max = 65536;      // LDS bytes one block may use
    int Fcap = 0;
    int cap_cells = 0;
    bool finished = false;
    bool profiling = false;
    // profiling: five events per batch (batch start, real-pass evaluation
    // start/end, random-pass evaluation start/end), recorded without a host
    // wait and resolved when the statistics are read
    std::vector<std::array<hipEvent_t, 5>> prof_ev;
    size_t prof_used = 0, prof_done = 0;
    std::vector<char> prof_random;                     // the batch had random passes
    std::vector<std::pair<float, float>> launch_ms;   // per batch: real, random evaluation (ms; -1 when absent)
    hipEvent_t rb_ev[RB_PIECES + 1] = {};   // pipelined read-back (cm_job_finish)
    double eval_ms = 0.0, total_ms = 0.0;
    int64_t eval_launches = 0, total_launches = 0, frames = 0;
    std::vector<Geo> hgeo;
    std::vector<int> huk, hdp, hdi;
    std::vector<int32_t> hgm;        // group maps (host copy of the upload)
    PinBuf hres;                     // accumulators and hit counts read back at finish (page-locked)
    // verification mode: every batch's records, placements and reference
    // draws are copied to the host, keyed by trajectory frame number
    bool verify = false;
    DevBuf vrec;
    struct VerifyFrame {
        std::vector<VRec> rec;            // [NP][Mv] (tiles family)
        std::vector<double> placed;       // [K][Nv][3], NaN where a slot was not placed
        std::vector<uint8_t> placed_flag; // [K][Mv]
        std::vector<int32_t> draws;       // [K]
    };
    std::map<int64_t, VerifyFrame> vstore;
    // buffers carved from a fixed device region instead of allocated (the
    // entry point that allocates nothing); null for ordinary jobs
    char* arena = nullptr;
    size_t arena_cap = 0, arena_used = 0;
};

namespace {

// Grows a job buffer.  A block being replaced may still be read by work
// queued on the job's stream: the host waits for that stream only (not the
// device, as hipFree would, which would stall the other slots of a request
// server), then the block goes back to the cache for later jobs.  Jobs with
// an arena take the next 256-byte aligned piece of it instead (never given
// back; the arena is reset per call).
int ensure(cm_job* J, DevBuf& b, size_t bytes)
{
    if (bytes == 0) bytes = 16;
    if (b.bytes >= bytes) return CM_OK;
    if (J->arena) {
        const size_t off = (J->arena_used + 255) & ~(size_t)255;
        if (off > J->arena_cap || bytes > J->arena_cap - off)
            return fail(CM_ENOMEM, "job does not fit the fixed device scratch of the no-allocation entry point");
        b.p = J->arena + off;
        b.bytes = bytes;
        J->arena_used = off + bytes;
        return CM_OK;
    }
    if (b.p) {
        if (J->stream) {
            const hipError_t e = hipStreamSynchronize(J->stream);
            if (e != hipSuccess) return fail(CM_EHIP, std::string("hipStreamSynchronize: ") + hipGetErrorString(e));
        }
        dev_put(b);
    }
    b.p = nullptr;
    b.bytes = 0;
    return dev_take(b, bytes);
}

// Layout of the buffers of the molecule pairs on the matrix cores for F
// frames; with base, their pointers.  Returns the bytes.
size_t cl_layout(const KP& P, int64_t F, char* base, Bufs* B)
{
    size_t o = 0;
    auto take = [&](size_t bytes) {
        char* p = base ? base + o : nullptr;
        o += (bytes + 255) & ~(size_t)255;
        return p;
    };
    // the key counts first: cleared together per batch
    ClSide cl[2] = {};
    const int sides = P.self_ ? 1 : 2;
    for (int k = 0; k < sides; k++) {
        cl[k].M = k ? P.Mv : P.Mu;
        cl[k].n = k ? P.nv : P.nu;
        while (((int64_t)4 << (3 * cl[k].bits)) < cl[k].M && cl[k].bits < 9) cl[k].bits++;
        cl[k].cnt = (int*)take((size_t)F << (3 * cl[k].bits) << 2);
    }
    const size_t zero = o;
    for (int k = 0; k < sides; k++) {
        cl[k].start = (int*)take((size_t)F << (3 * cl[k].bits) << 2);
        cl[k].key = (int*)take((size_t)4 * F * cl[k].M);
        cl[k].rank = (int*)take((size_t)4 * F * cl[k].M);
        cl[k].ord = (int*)take((size_t)4 * F * cl[k].M);
        cl[k].cen = (double*)take((size_t)24 * F * cl[k].M);
    }
    float* a = (float*)take((size_t)256 * F * P.nT);
    float* b = (float*)take((size_t)256 * F * P.nB * P.nv);
    float4* ti = (float4*)take((size_t)48 * F * P.nT);
    float4* bi = (float4*)take((size_t)48 * F * P.nB);
    float4* si = (float4*)take((size_t)32 * F * P.nS);
    if (B) {
        B->cl[0] = cl[0]; B->cl[1] = cl[1];
        B->clA = a; B->clB = b; B->tinfo = ti; B->binfo = bi; B->sinfo = si;
    }
    return base ? zero : o;
}

int64_t per_frame_bytes(const cm_job* J, int dtype_size, bool host_input, int64_t cap, int64_t kcap)
{
    int64_t Mu = J->d.nmols_u, Mv = J->d.nmols_v, NP = 1 + J->K;
    int64_t b = sizeof(Geo) + 64;
    if (host_input) b += (J->Nu + J->Nv) * 3 * dtype_size;
    int64_t items = J->atoms_family ? J->d.natoms_per_mol_u : Mu;
    if (!J->kp.rpm) b += items * (16 + 16 + 4) + (cap + 1) * 8;
    if (!J->atoms_family) {
        b += J->Nu * 16 + Mu * 16 + (Mu + 1) * 4 + J->K * 8;
        b += J->kp.rpm ? (int64_t)cl_layout(J->kp, 1, nullptr, nullptr) : J->Nv * 16 + Mv * 20;
        b += (int64_t)J->K * (J->Nv * (24 + 16) + Mv * 16);
    } else {
        b += cap * 9 + NP * ((kcap + 1) * 8 + Mv * 12 + 4) + 8;
        b += J->Nv * 16 + (int64_t)J->K * J->Nv * (24 + 16);
    }
    b += (int64_t)J->kb * Mv * 5 + J->kb * 4;
    return b;
}

int64_t cells_for(const cm_job* J, const double* cell9, int64_t* keys)
{
    cm::Cell64 c;
    cm::cell_setup(cell9, J->d.triclinic, &c);
    double sp[3];
    plane_spacings(c.H, sp);
    double side = J->atoms_family ? J->kp.cutsys * J->cell_frac : J->kp.cutsys;
    int64_t n = 1, mx = 1;
    for (int k = 0; k < 3; k++) {
        int64_t nk = std::max<int64_t>(1, (int64_t)std::floor(sp[k] / side));
        n *= nk;
        mx = std::max(mx, nk);
    }
    int bits = 0;
    while (((int64_t)1 << bits) < mx) bits++;
    *keys = (int64_t)1 << (3 * bits);
    return n;
}

// tiles of 16 columns an evaluating wavefront holds (eval_chunk's G): molecules
// of three atoms, or atoms
int chunk_groups(const KP& P, bool random)
{
    const int mpt = random ? P.mpt_r : P.mpt;
    if (P.mol_lane) return mpt > 32 ? 4 : (mpt > 16 ? 2 : 1);
    return mpt > lane_molecules(P.nv) ? 8 : 4;
}

// Wavefronts per block of an evaluation and its LDS: as many (up to 16) as fit
// one CU's LDS together with the histograms and the chunk table
struct EvShape {
    int waves;
    size_t lds;
    EvShape(const KP& P, int G, int TQ, int table, int lds_max)
    {
        const size_t head = 4 * (((size_t)EvHist::words(P) + table + 3) & ~(size_t)3), per = 4 * (size_t)eval_wave_words(G, TQ);
        waves = (int)std::max<int64_t>(1, std::min<int64_t>(16, ((int64_t)lds_max - (int64_t)head) / (int64_t)per));
        lds = head + per * waves;
    }
};

int lds_per_block(int dev)
{
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v < 65536) v = 65536;
    return v;
}

// grid 0: as many workgroups as the device holds at once (persistent kernel)
template <class TU, class TV, bool RANDOM, int G, int TQ>
void launch_tiles_one(hipStream_t s, int grid, const cm_job* J, const KP& P, const Bufs& B, const void* xu, const void* xv)
{
    const int nfp = P.F * (RANDOM ? P.NG : 1);
    const EvShape sh(P, G, TQ, nfp + 1 <= CBCAP ? nfp + 1 : 0, J->lds_max);
    // verification (records kept) in its own instantiations, so that the
    // ordinary kernels carry none of its registers
    auto kern = B.vrec ? k_eval_tiles<TU, TV, RANDOM, G, TQ, true> : k_eval_tiles<TU, TV, RANDOM, G, TQ, false>;
    if (grid <= 0) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, 64 * sh.waves, sh.lds) != hipSuccess || nb < 1) nb = 1;
        grid = nb * J->cus;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * sh.waves), sh.lds, s, P, B, (const TU*)xu, (const TV*)xv);
    auto res = B.vrec ? k_resolve<TU, TV, RANDOM, true> : k_resolve<TU, TV, RANDOM, false>;
    hipLaunchKernelGGL(res, dim3((unsigned)resolve_parts(P, RANDOM), (unsigned)std::min(nfp, 65535)), dim3(BLOCK), 0, s, P, B,
                       (const TU*)xu, (const TV*)xv);
}

template <class TU, class TV, bool RANDOM>
void launch_tiles(hipStream_t s, int grid, const cm_job* J, const KP& P, const Bufs& B, const void* xu, const void* xv)
{
    const int g = chunk_groups(P, RANDOM);
    if (P.mol_lane) {
        if (g == 4) launch_tiles_one<TU, TV, RANDOM, 4, 3>(s, grid, J, P, B, xu, xv);
        else if (g == 2) launch_tiles_one<TU, TV, RANDOM, 2, 3>(s, grid, J, P, B, xu, xv);
        else launch_tiles_one<TU, TV, RANDOM, 1, 3>(s, grid, J, P, B, xu, xv);
    } else {
        if (g == 8) launch_tiles_one<TU, TV, RANDOM, 8, ATOMS>(s, grid, J, P, B, xu, xv);
        else launch_tiles_one<TU, TV, RANDOM, 4, ATOMS>(s, grid, J, P, B, xu, xv);
    }
}

void launch_tiles_any(bool f32, bool random, hipStream_t s, int grid, const cm_job* J, const KP& P, const Bufs& B,
                      const void* xu, const void* xv)
{
    if (f32) {
        if (random) launch_tiles<float, float, true>(s, grid, J, P, B, xu, xv);
        else launch_tiles<float, float, false>(s, grid, J, P, B, xu, xv);
    } else {
        if (random) launch_tiles<double, double, true>(s, grid, J, P, B, xu, xv);
        else launch_tiles<double, double, false>(s, grid, J, P, B, xu, xv);
    }
}

// Verification mode: waits for the batch and keeps, per frame, the records
// of every pass (tiles family), the placed solvent of every random pass (by
// slot) and the drawn reference solute molecules.
int verify_collect(cm_job* J, int F, const int64_t* frame_index)
{
    HIPCHK(hipStreamSynchronize(J->stream));
    const int64_t Mv = J->d.nmols_v, Nv = J->Nv, K = J->K, NP = 1 + K, nv = J->d.natoms_per_mol_v;
    std::vector<VRec> rec;
    if (J->atoms_family) {
        rec.resize((size_t)F * NP * Mv);
        HIPCHK(hipMemcpy(rec.data(), J->vrec.p, sizeof(VRec) * rec.size(), hipMemcpyDeviceToHost));
    }
    std::vector<double> P;
    std::vector<int> msorted, nnear;
    if (K > 0) {
        P.resize((size_t)F * K * Nv * 3);
        HIPCHK(hipMemcpy(P.data(), J->P.p, sizeof(double) * P.size(), hipMemcpyDeviceToHost));
        if (J->atoms_family) {
            msorted.resize((size_t)F * NP * Mv);
            nnear.resize((size_t)F * (1 + J->kp.NG));
            HIPCHK(hipMemcpy(msorted.data(), J->msorted.p, sizeof(int) * msorted.size(), hipMemcpyDeviceToHost));
            HIPCHK(hipMemcpy(nnear.data(), J->nnear.p, sizeof(int) * nnear.size(), hipMemcpyDeviceToHost));
        }
    }
    for (int f = 0; f < F; f++) {
        cm_job::VerifyFrame& vf = J->vstore[frame_index[f]];
        if (J->atoms_family) vf.rec.assign(rec.begin() + (size_t)f * NP * Mv, rec.begin() + (size_t)(f + 1) * NP * Mv);
        vf.placed.assign((size_t)K * Nv * 3, NAN);
        vf.placed_flag.assign((size_t)K * Mv, 0);
        vf.draws.assign((size_t)K, 0);
        if (J->atoms_family) {
            // near slots only, stored at their sorted positions within their group
            const int64_t KM = J->kp.KM, NG = J->kp.NG;
            for (int64_t grp = 0; grp < (K > 0 ? NG : 0); grp++) {
                const double* src = P.data() + ((size_t)f * K + grp * KM) * Nv * 3;
                const int* ms = msorted.data() + ((size_t)f * NP + 1 + grp * KM) * Mv;
                for (int64_t pos = 0; pos < nnear[f * (1 + NG) + 1 + grp]; pos++) {
                    const int64_t slot = grp * KM * Mv + ms[pos];   // pass times Mv plus the molecule
                    std::memcpy(vf.placed.data() + slot * nv * 3, src + pos * nv * 3, sizeof(double) * 3 * nv);
                    vf.placed_flag[slot] = 1;
                }
            }
            continue;
        }
        for (int64_t k = 0; k < K; k++) {
            std::memcpy(vf.placed.data() + (size_t)k * Nv * 3, P.data() + ((size_t)f * K + k) * Nv * 3, sizeof(double) * 3 * Nv);
            std::fill(vf.placed_flag.begin() + k * Mv, vf.placed_flag.begin() + (k + 1) * Mv, (uint8_t)1);
            vf.draws[k] = J->huk[(size_t)f * K + k];
        }
    }
    return CM_OK;
}

// Host geometry of a batch's frames: cells, inverses, plane spacings and, for
// the single-solute kernels, the fine cell grid.
int batch_geo(const cm_job* J, int F, const int64_t* frame_index, const double* cells, int64_t cap, int64_t kcap, Geo* out)
{
    const double cutsys = J->kp.cutsys;
    for (int f = 0; f < F; f++) {
        Geo& g = out[f];
        memset(&g, 0, sizeof(Geo));
        cm::cell_setup(cells + 9 * f, J->d.triclinic, &g.cell);
        for (int k = 0; k < 9; k++) {
            g.H32[k] = (float)g.cell.H[k];
            g.Hi32[k] = (float)g.cell.Hi[k];
        }
        plane_spacings(g.cell.H, g.sp);
        g.ortho = (g.cell.H[1] == 0.0 && g.cell.H[2] == 0.0 && g.cell.H[3] == 0.0 && g.cell.H[5] == 0.0 &&
                   g.cell.H[6] == 0.0 && g.cell.H[7] == 0.0) ? 1 : 0;
        double spmin = std::min(g.sp[0], std::min(g.sp[1], g.sp[2]));
        if (!(cutsys < 0.5 * spmin * (1.0 - 1e-9)))
            return fail(CM_EUNSUPPORTED, "cutoff must be smaller than half of the smallest plane spacing of the unit cell");
        g.frame = (uint32_t)frame_index[f];
        if (J->atoms_family) {
            double side = cutsys * J->cell_frac;
            g.ncell = 1;
            for (int k = 0; k < 3; k++) {
                g.nc[k] = std::max(1, (int)std::floor(g.sp[k] / side));
                g.ncell *= g.nc[k];
            }
            if (g.ncell > cap) return fail(CM_EHIP, "internal error: fine grid larger than its allocation");
            int mx = std::max(g.nc[0], std::max(g.nc[1], g.nc[2]));
            g.kbits = 0;
            while ((1 << g.kbits) < mx) g.kbits++;
            if ((int64_t)1 << (3 * g.kbits) > kcap) return fail(CM_EHIP, "internal error: key space larger than its allocation");
        }
    }
    return CM_OK;
}

// The kernels' view of a job's buffers (geometry array at geo)
// The near flags [F][cap] (bytes) and, after them, the encoded distances of
// the cell centres [F][cap] and lower corners [F][cap] of the tiles family:
// one block, cleared together per batch.
size_t near_flags_bytes(int64_t F, int64_t cap) { return ((size_t)F * cap + 15) & ~(size_t)15; }
size_t near_bytes(int64_t F, int64_t cap) { return near_flags_bytes(F, cap) + (((size_t)8 * F * cap + 15) & ~(size_t)15); }

Bufs batch_bufs(const cm_job* J, Geo* geo)
{
    Bufs B;
    memset(&B, 0, sizeof(B));
    B.geo = geo;
    B.cnt = (int*)J->cells_cnt.p;
    B.start = (int*)J->cells_start.p;
    B.tmp4 = (float4*)J->tmp4.p;
    B.tmpcell = (int*)J->tmpcell.p;
    B.sorted = (float4*)J->sorted.p;
    B.nitems = J->atoms_family ? J->kp.nu : J->kp.Mu;
    B.solw = (float4*)J->solw.p;
    B.ucen = (float4*)J->ucen.p;
    B.vw = (float4*)J->vw.p;
    B.vcell = (int*)J->vcell.p;
    B.vcen = (float4*)J->vcen.p;
    B.P = (double*)J->P.p;
    B.vw_r = (float4*)J->vw_r.p;
    B.vcen_r = (float4*)J->vcen_r.p;
    B.bflag = (unsigned char*)J->bflag.p;
    B.blist = (int*)J->blist.p;
    B.nbulk = (int*)J->nbulk.p;
    B.uk = (int*)J->uk.p;
    B.drawn_ptr = (int*)J->drawn_ptr.p;
    B.drawn_idx = (int*)J->drawn_idx.p;
    B.near = (unsigned char*)J->near.p;
    B.mkey = (int*)J->mkey.p;
    B.mrank = (int*)J->mrank.p;
    B.mcnt = (int*)J->mcnt.p;
    B.mstart = (int*)J->mstart.p;
    B.msum = (int*)J->msum.p;
    B.resmask = (unsigned*)J->mkey.p;
    B.msorted = (int*)J->msorted.p;
    B.nnear = (int*)J->nnear.p;
    B.chunk_base = (int*)J->chunk_base.p;
    ull* c = (ull*)J->cnt.p;
    const int64_t nb = J->d.nbins, ngu = J->d.n_groups_u, ngv = J->d.n_groups_v;
    B.cnt_md = c; B.cnt_md_r = c + nb; B.cnt_rdf = c + 2 * nb; B.cnt_rdf_r = c + 3 * nb;
    B.cnt_gu = c + 4 * nb; B.cnt_gv = B.cnt_gu + ngu * nb; B.cnt_gu_r = B.cnt_gv + ngv * nb; B.cnt_gv_r = B.cnt_gu_r + ngu * nb;
    B.stats = (ull*)J->stats.p;
    return B;
}

// bytes of the key counts of a batch (and of the keys' starts)
size_t key_bytes(const KP& P, int F) { return sizeof(int) * (size_t)F * ((size_t)P.kcap + (size_t)P.NG * P.kcapr); }

// scan of the key counts of the real pass (random 0) or the random groups of a batch
void launch_scan(hipStream_t s, const KP& P, const Bufs& B, int random)
{
    const int parts = scan_parts(random ? P.kcapr : P.kcap);
    const dim3 gr((unsigned)parts, (unsigned)(P.F * (random ? P.NG : 1)));
    if (parts > 1) hipLaunchKernelGGL(k_scan_sums, gr, dim3(1024), 0, s, P, B, random);
    hipLaunchKernelGGL(k_scan_rows, gr, dim3(1024), 0, s, P, B, random);
}

// molecule pairs on the matrix cores: order, operands and boxes of a batch
template <class T>
void launch_cl_prep(hipStream_t s, const KP& P, const Bufs& B, const void* xu, const void* xv)
{
    const unsigned sides = P.self_ ? 1 : 2, F = (unsigned)P.F;
    const int64_t M = P.self_ ? P.Mu : std::max(P.Mu, P.Mv);
    const unsigned gm = (unsigned)((M + BLOCK - 1) / BLOCK);
    hipLaunchKernelGGL(k_cl_keys<T>, dim3(std::min(gm, 64u), F, sides), dim3(BLOCK), 0, s, P, B, (const T*)xu, (const T*)xv);
    hipLaunchKernelGGL(k_cl_scan, dim3(F, sides), dim3(1024), 0, s, P, B);
    hipLaunchKernelGGL(k_cl_order, dim3(grid_for(M * F), sides), dim3(BLOCK), 0, s, P, B);
    const unsigned gb = (unsigned)std::max(P.nS, (P.nB + BLOCK / 64 - 1) / (BLOCK / 64));
    hipLaunchKernelGGL(k_cl_build<T>, dim3(gb, F, 2), dim3(BLOCK), 0, s, P, B,
                       (const T*)xu, (const T*)xv);
}

template <class T, int RPM, int NVT, bool SELF>
void launch_cl_one(hipStream_t s, const cm_job* J, const KP& P, const Bufs& B, const void* xu, const void* xv)
{
    auto kern = k_cl_eval<T, T, RPM, NVT, SELF>;
    const int gwords = P.glds ? P.nbins * (P.gnu + (P.self_ ? 0 : P.gnv)) : 0;
    const int64_t head = 4 * (int64_t)((2 * P.nbins + gwords + 3) & ~3);
    const int waves = (int)std::max<int64_t>(1, std::min<int64_t>(NVT > 8 ? 8 : 16, (J->lds_max - head) / (4 * CL_WORDS)));
    const size_t lds = (size_t)(head + 4 * (int64_t)CL_WORDS * waves);
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, 64 * waves, lds) != hipSuccess || nb < 1) nb = 1;
    // Few clusters: S wavefronts split a cluster's tiles, so that every wavefront
    // of the device has about two items of four tiles or more; beyond 16 by super
    // tiles first, eight or more each (a wavefront tests the tiles of its own only;
    // below, the tiles divide more evenly).  Ten frames of 40 ions in 8,000 waters,
    // 30 clusters of up to 2,000 tiles: 249 us with 16 wavefronts a cluster, 76 us
    // so; 2,000 waters, 10 frames, 1,250 clusters: 132 us with six by tiles, 144
    // with four by super tiles and two by tiles.
    const int64_t items = (int64_t)P.F * P.nB, want = 2 * (int64_t)nb * J->cus * waves;
    const int64_t most = std::max(P.nT / 4, std::min(16, P.nT));
    const int S0 = (int)std::min<int64_t>(most, std::max<int64_t>(1, want / std::max<int64_t>(items, 1)));
    const int Sg = std::min((S0 + 15) / 16, std::max(1, P.nS / 8)), S = (S0 + Sg - 1) / Sg * Sg;
    const int64_t blocks = std::min<int64_t>((int64_t)nb * J->cus, (items * S + waves - 1) / waves);
    hipLaunchKernelGGL(kern, dim3((unsigned)((blocks + 7) / 8 * 8)), dim3(64 * waves), lds, s, P, B, (const T*)xu, (const T*)xv, S, Sg);
}

template <class T, int RPM>
void launch_cl_rpm(hipStream_t s, const cm_job* J, const KP& P, const Bufs& B, const void* xu, const void* xv)
{
    if (P.self_) {
        // the same molecules on both sides
        if (RPM == 4 && P.nv == 3) launch_cl_one<T, RPM, RPM == 4 ? 3 : RPM, true>(s, J, P, B, xu, xv);
        else launch_cl_one<T, RPM, RPM, true>(s, J, P, B, xu, xv);
    } else {
        if (P.nv == 3) launch_cl_one<T, RPM, 3, false>(s, J, P, B, xu, xv);
        else if (P.nv <= 4) launch_cl_one<T, RPM, 4, false>(s, J, P, B, xu, xv);
        else if (P.nv <= 8) launch_cl_one<T, RPM, 8, false>(s, J, P, B, xu, xv);
        else launch_cl_one<T, RPM, 16, false>(s, J, P, B, xu, xv);
    }
}

template <class T>
void launch_cl(hipStream_t s, const cm_job* J, const KP& P, const Bufs& B, const void* xu, const void* xv)
{
    if (P.rpm == 1) {
        if (P.self_) launch_cl_one<T, 1, 1, true>(s, J, P, B, xu, xv);
        else launch_cl_one<T, 1, 1, false>(s, J, P, B, xu, xv);
    } else if (P.rpm == 4) launch_cl_rpm<T, 4>(s, J, P, B, xu, xv);
    else if (P.rpm == 8) launch_cl_rpm<T, 8>(s, J, P, B, xu, xv);
    else launch_cl_rpm<T, 16>(s, J, P, B, xu, xv);
}

void launch_cl_any(hipStream_t s, const cm_job* J, const KP& P, const Bufs& B, bool f32, const void* xu, const void* xv)
{
    if (f32) launch_cl<float>(s, J, P, B, xu, xv);
    else launch_cl<double>(s, J, P, B, xu, xv);
}

int run_batch(cm_job* J, int F, const int64_t* frame_index, const void* xu_dev, const void* xv_dev, int dtype,
              const double* cells, int64_t cap, int64_t kcap)
{
    KP P = J->kp;
    P.F = F;
    P.cap = (int)cap;
    P.kcap = (int)kcap;
    P.kcapr = (int)(kcap << (3 * P.ksub));
    P.mpt_auto = chunks_vary(P) ? 1 : 0;
    const bool tiles = J->atoms_family;
    // geometry on the host: cells, inverse, spacings (and the fine grid of the tiles family)
    J->hgeo.assign(F, Geo());
    if (int r = batch_geo(J, F, frame_index, cells, cap, kcap, J->hgeo.data())) return r;
    hipStream_t s = J->stream;
    HIPCHK(hipMemcpyAsync(J->geo.p, J->hgeo.data(), sizeof(Geo) * F, hipMemcpyHostToDevice, s));
    Bufs B = batch_bufs(J, (Geo*)J->geo.p);
    B.dfield = (unsigned*)((char*)J->near.p + near_flags_bytes(F, cap));
    B.vrec = (J->verify && tiles) ? (VRec*)J->vrec.p : nullptr;
    if (B.vrec) {
        const int64_t nrec = (int64_t)F * P.NP * P.Mv;
        hipLaunchKernelGGL(k_vrec_init, dim3(grid_for(nrec)), dim3(BLOCK), 0, s, B.vrec, nrec);
    }

    FillList fills;
    // random draws of the reference solute molecules (mddf_frame!, src/mddf.jl:374-376);
    // with one solute molecule every draw is molecule 0
    if (!tiles && J->K > 0) {
        J->huk.assign((size_t)F * J->K, 0);
        J->hdp.assign((size_t)F * (P.Mu + 1), 0);
        J->hdi.assign((size_t)F * J->K, 0);
        for (int f = 0; f < F; f++) {
            int* dp = &J->hdp[(size_t)f * (P.Mu + 1)];
            for (int k = 0; k < J->K; k++) {
                cm::u32x4 r = cm::philox4x32_10({(uint32_t)k, 0u, (uint32_t)frame_index[f], cm::TAG_REF}, P.key0, P.key1);
                int u = (int)cm::draw_index(r.x, P.Mu);
                J->huk[(size_t)f * J->K + k] = u;
                dp[u + 1]++;
            }
            for (int u = 0; u < P.Mu; u++) dp[u + 1] += dp[u];
            std::vector<int> fill(P.Mu, 0);
            for (int k = 0; k < J->K; k++) {
                int u = J->huk[(size_t)f * J->K + k];
                J->hdi[(size_t)f * J->K + dp[u] + fill[u]++] = k;
            }
        }
        HIPCHK(hipMemcpyAsync(J->uk.p, J->huk.data(), sizeof(int) * J->huk.size(), hipMemcpyHostToDevice, s));
        HIPCHK(hipMemcpyAsync(J->drawn_ptr.p, J->hdp.data(), sizeof(int) * J->hdp.size(), hipMemcpyHostToDevice, s));
        HIPCHK(hipMemcpyAsync(J->drawn_idx.p, J->hdi.data(), sizeof(int) * J->hdi.size(), hipMemcpyHostToDevice, s));
    } else if (J->K > 0) {
        fills.add(J->uk.p, sizeof(int) * (size_t)F * J->K);
    }
    if (P.rpm) {
        const size_t zero = cl_layout(P, F, (char*)J->clmem.p, &B);
        fills.add(J->clmem.p, zero);
    } else fills.add(J->cells_cnt.p, sizeof(int) * (size_t)F * (cap + 1));
    if (tiles) {
        fills.add(J->near.p, near_bytes(F, cap));
        fills.add(J->mcnt.p, key_bytes(P, F));
        // the bulk flags' start (k_bulk_init without a molecule to leave out)
        if (P.K > 0) fills.add(J->bflag.p, (size_t)F * P.kb * P.Mv, P.usecutoff ? 0u : 0x01010101u);
    }
    if (int r = fill_async(fills, s)) return r;

    const bool f32 = dtype == CM_F32;
    const float* uf = (const float*)xu_dev;
    const float* vf = (const float*)xv_dev;
    const double* ud = (const double*)xu_dev;
    const double* vd = (const double*)xv_dev;
    const size_t shm = sizeof(unsigned) * 2 * P.nbins;
    hipEvent_t ev[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    if (J->profiling) {
        if (J->prof_used == J->prof_ev.size()) {
            std::array<hipEvent_t, 5> a{};
            for (auto& e : a) HIPCHK(hipEventCreate(&e));
            J->prof_ev.push_back(a);
        }
        for (int k = 0; k < 5; k++) ev[k] = J->prof_ev[J->prof_used][k];
        J->prof_used++;
        HIPCHK(hipEventRecord(ev[4], s));
        J->prof_random.push_back(P.K > 0 ? 1 : 0);
    }
    const int mols = tiles ? 0 : 1;
    if (!P.rpm) {
        {
            const int64_t nm = (int64_t)P.Mv + (mols ? P.Mu : 0);
            const dim3 gr((unsigned)std::min<int64_t>((nm + BLOCK - 1) / BLOCK, 64), (unsigned)F);
            if (f32) hipLaunchKernelGGL(k_radii<float>, gr, dim3(BLOCK), 0, s, P, B, uf, vf, mols);
            else hipLaunchKernelGGL(k_radii<double>, gr, dim3(BLOCK), 0, s, P, B, ud, vd, mols);
        }
    }
    if (P.rpm) {
        if (f32) launch_cl_prep<float>(s, P, B, xu_dev, xv_dev);
        else launch_cl_prep<double>(s, P, B, xu_dev, xv_dev);
    } else {
        if (tiles) {
            int64_t n = (int64_t)F * P.nu;
            if (f32) hipLaunchKernelGGL(k_wrap_atoms<float>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, uf);
            else hipLaunchKernelGGL(k_wrap_atoms<double>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, ud);
        } else {
            int64_t n = (int64_t)F * P.Mu;
            if (f32) hipLaunchKernelGGL(k_prep_solute_mols<float>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, uf);
            else hipLaunchKernelGGL(k_prep_solute_mols<double>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, ud);
        }
        hipLaunchKernelGGL(k_scan_cells, dim3(F), dim3(1024), 0, s, P, B);
        hipLaunchKernelGGL(k_scatter, dim3(grid_for((int64_t)F * B.nitems)), dim3(BLOCK), 0, s, P, B, B.nitems);
        if (tiles) {
            hipLaunchKernelGGL(k_near_mark, dim3(near_blocks(P.nu), std::min(F, 65535)), dim3(BLOCK), 0, s, P, B);
            hipLaunchKernelGGL(k_dfield, dim3(grid_for((int64_t)F * cap * 16)), dim3(BLOCK), 0, s, P, B);
            int64_t n = (int64_t)F * P.Mv;
            if (f32) hipLaunchKernelGGL(k_prep_solvent_tiles<float>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, vf);
            else hipLaunchKernelGGL(k_prep_solvent_tiles<double>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, vd);
            launch_scan(s, P, B, 0);
            hipLaunchKernelGGL(k_mol_scatter, grid_slots(P.Mv, F), dim3(BLOCK), 0, s, P, B, 0);
            if (f32) hipLaunchKernelGGL(k_fill_real<float>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, vf);
            else hipLaunchKernelGGL(k_fill_real<double>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, vd);
            hipLaunchKernelGGL(P.mpt_auto ? k_chunk_table<true> : k_chunk_table<false>, dim3(1), dim3(1024), 0, s, P, B, 0);
        } else {
            int64_t n = (int64_t)F * P.Mv;
            if (f32) hipLaunchKernelGGL(k_prep_solvent<float>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, vf);
            else hipLaunchKernelGGL(k_prep_solvent<double>, dim3(grid_for(n)), dim3(BLOCK), 0, s, P, B, vd);
        }
    }
    if (P.K > 0 && !tiles) hipLaunchKernelGGL(k_bulk_init, dim3(grid_for((int64_t)F * P.kb * P.Mv)), dim3(BLOCK), 0, s, P, B);
    HIPCHK(hipGetLastError());
    // real pass
    if (J->profiling) HIPCHK(hipEventRecord(ev[0], s));
    if (tiles) {
        launch_tiles_any(f32, false, s, J->eval_grid, J, P, B, xu_dev, xv_dev);
    } else if (P.rpm) {
        launch_cl_any(s, J, P, B, f32, xu_dev, xv_dev);
    } else {
        int64_t n = (int64_t)F * P.Mv;
        const int gwords = P.glds ? P.nbins * (P.gnu + (P.self_ ? 0 : P.gnv)) : 0;
        const size_t shq = sizeof(unsigned) * ((2 * P.nbins + gwords + 3) & ~3) + sizeof(int4) * QCAP * (BLOCK / 64) +
                           (P.self_ ? sizeof(int4) * 2 * DCAP * (BLOCK / 64) : 0);
        // small systems: S lanes per solvent molecule split its neighbour walk
        // so that the launch still has about 6 wavefronts per SIMD of work
        const int64_t lanes = (int64_t)P.Mv * F;
        const int S = (int)std::min<int64_t>(14, std::max<int64_t>(1, (int64_t)(J->cus * 4 * 6 * 64) / std::max<int64_t>(lanes, 1)));
        const int gx = (int)std::max<int64_t>(1, std::min<int64_t>(((int64_t)P.Mv * S + BLOCK - 1) / BLOCK, 4096 / F + 1));
        const dim3 gr((unsigned)(8 * ((gx * F + 7) / 8)));
        // self-MDDF of 3- and 8-atom molecules (water, urea-like) keeps both
        // molecules of a pair in registers
        const int nfix = (P.self_ && P.nu == P.nv && (P.nu == 3 || P.nu == 8)) ? P.nu : 0;
        if (f32) {
            if (nfix == 3) hipLaunchKernelGGL((k_eval_mols_real<float, float, 3>), gr, dim3(BLOCK), shq, s, P, B, uf, vf, gx, S);
            else if (nfix == 8) hipLaunchKernelGGL((k_eval_mols_real<float, float, 8>), gr, dim3(BLOCK), shq, s, P, B, uf, vf, gx, S);
            else hipLaunchKernelGGL((k_eval_mols_real<float, float, 0>), gr, dim3(BLOCK), shq, s, P, B, uf, vf, gx, S);
        } else {
            if (nfix == 3) hipLaunchKernelGGL((k_eval_mols_real<double, double, 3>), gr, dim3(BLOCK), shq, s, P, B, ud, vd, gx, S);
            else if (nfix == 8) hipLaunchKernelGGL((k_eval_mols_real<double, double, 8>), gr, dim3(BLOCK), shq, s, P, B, ud, vd, gx, S);
            else hipLaunchKernelGGL((k_eval_mols_real<double, double, 0>), gr, dim3(BLOCK), shq, s, P, B, ud, vd, gx, S);
        }
    }
    if (J->profiling) HIPCHK(hipEventRecord(ev[1], s));
    HIPCHK(hipGetLastError());
    // random passes
    if (P.K > 0) {
        hipLaunchKernelGGL(k_bulk_compact, dim3(F * P.kb), dim3(1024), 0, s, P, B, tiles ? 0 : 1);
        if (tiles) {
            hipLaunchKernelGGL(k_place_keys, grid_slots(P.Mv, F * P.K), dim3(BLOCK), 0, s, P, B);
            launch_scan(s, P, B, 1);
            const dim3 gs = grid_slots(P.KM * P.Mv, F * P.NG);
            hipLaunchKernelGGL(k_mol_scatter, gs, dim3(BLOCK), 0, s, P, B, 1);
            if (f32) hipLaunchKernelGGL(k_place_near<float>, gs, dim3(BLOCK), 0, s, P, B, vf);
            else hipLaunchKernelGGL(k_place_near<double>, gs, dim3(BLOCK), 0, s, P, B, vd);
            hipLaunchKernelGGL(P.mpt_auto ? k_chunk_table<true> : k_chunk_table<false>, dim3(1), dim3(1024), 0, s, P, B, 1);
        } else {
            hipLaunchKernelGGL(k_mols_near, grid_slots((P.Mv + NEAR_SLOTS - 1) / NEAR_SLOTS, F * P.K), dim3(BLOCK), 0, s, P, B);
        }
        HIPCHK(hipGetLastError());
        if (J->profiling) HIPCHK(hipEventRecord(ev[2], s));
        if (tiles) {
            launch_tiles_any(f32, true, s, J->eval_grid, J, P, B, xu_dev, xv_dev);
        } else {
            const int gwords = P.glds ? P.nbins * (P.gnu + (P.self_ ? 0 : P.gnv)) : 0;
            const size_t shr = sizeof(unsigned) * (2 * P.nbins + gwords);
            // about four blocks per CU; pairs of their own where there are enough
            const int64_t fk = (int64_t)F * P.K, want = 4 * (int64_t)J->cus;
            const unsigned gy = (unsigned)std::min<int64_t>(fk, want);
            const unsigned gx = (unsigned)std::max<int64_t>(1, std::min<int64_t>((P.Mv + BLOCK - 1) / BLOCK, want / gy));
            if (f32) hipLaunchKernelGGL((k_eval_mols_rand<float, float>), dim3(gx, gy), dim3(BLOCK), shr, s, P, B, uf, vf);
            else hipLaunchKernelGGL((k_eval_mols_rand<double, double>), dim3(gx, gy), dim3(BLOCK), shr, s, P, B, ud, vd);
        }
        if (J->profiling) HIPCHK(hipEventRecord(ev[3], s));
    }
    // (geometry errors detected on the device are in the job's error bits and
    // reported when the job is collected: the host does not wait for the batch
    // here and prepares the next one while it runs)
    HIPCHK(hipGetLastError());
    J->frames += F;
    if (J->verify) return verify_collect(J, F, frame_index);
    return CM_OK;
}

// sizes of the buffers cleared per batch, rounded up to whole 16-byte words
// (the multi-job path clears them with 16-byte stores)
size_t round16(size_t b) { return (b + 15) & ~(size_t)15; }

int alloc_batch(cm_job* J, int F, int64_t cap, int64_t kcap, int dtype_size, bool host_input)
{
    int r;
    int64_t Mu = J->d.nmols_u, Mv = J->d.nmols_v, NP = 1 + J->K;
    int64_t items = J->atoms_family ? J->d.natoms_per_mol_u : Mu;
    if ((r = ensure(J, J->geo, sizeof(Geo) * F))) return r;
    const bool cl = J->kp.rpm > 0;
    if (cl) {
        if ((r = ensure(J, J->clmem, cl_layout(J->kp, F, nullptr, nullptr)))) return r;
    } else {
        if ((r = ensure(J, J->cells_cnt, round16(sizeof(int) * F * (cap + 1))))) return r;
        if ((r = ensure(J, J->cells_start, sizeof(int) * F * (cap + 1)))) return r;
        if ((r = ensure(J, J->tmp4, 16 * F * items))) return r;
        if ((r = ensure(J, J->tmpcell, 4 * F * items))) return r;
        if ((r = ensure(J, J->sorted, 16 * F * items))) return r;
        if ((r = ensure(J, J->vw, 16 * F * J->Nv))) return r;
    }
    if (!J->atoms_family) {
        if ((r = ensure(J, J->solw, 16 * F * J->Nu))) return r;
        if ((r = ensure(J, J->ucen, 16 * F * Mu))) return r;
        if ((r = ensure(J, J->drawn_ptr, 4 * F * (Mu + 1)))) return r;
        if ((r = ensure(J, J->drawn_idx, 4 * F * std::max(J->K, 1)))) return r;
        if (!cl) {
            if ((r = ensure(J, J->vcell, 4 * F * Mv))) return r;
            if ((r = ensure(J, J->vcen, 16 * F * Mv))) return r;
        }
    } else {
        if ((r = ensure(J, J->near, near_bytes(F, cap)))) return r;
        // (also the chunks' resmask: four bytes, eight in chunks of more than 32
        // molecules; a row may end in a chunk of fewer)
        if ((r = ensure(J, J->mkey, (size_t)4 * F * NP * Mv + (size_t)8 * F * (1 + J->kp.NG)))) return r;
        if ((r = ensure(J, J->mrank, (size_t)4 * F * NP * Mv))) return r;
        KP P = J->kp;
        P.kcap = (int)kcap;
        P.kcapr = (int)(kcap << (3 * P.ksub));
        if ((r = ensure(J, J->mcnt, round16(key_bytes(P, F))))) return r;
        if ((r = ensure(J, J->mstart, key_bytes(P, F)))) return r;
        if ((r = ensure(J, J->msum, (size_t)4 * F * (scan_parts(P.kcap) + P.NG * scan_parts(P.kcapr))))) return r;
        if ((r = ensure(J, J->msorted, (size_t)4 * F * NP * Mv))) return r;
        if ((r = ensure(J, J->nnear, (size_t)4 * F * (1 + P.NG)))) return r;
        if ((r = ensure(J, J->chunk_base, (size_t)4 * (F * std::max(J->K, 1) + MPT_AT + 1)))) return r;
    }
    if (J->K > 0) {
        if ((r = ensure(J, J->P, (size_t)24 * F * J->K * J->Nv))) return r;
        if ((r = ensure(J, J->vw_r, (size_t)16 * F * J->K * J->Nv))) return r;
        if (!J->atoms_family) {
            if ((r = ensure(J, J->vcen_r, (size_t)16 * F * J->K * Mv))) return r;
        }
        if ((r = ensure(J, J->bflag, (size_t)F * J->kb * Mv))) return r;
        if ((r = ensure(J, J->blist, (size_t)4 * F * J->kb * Mv))) return r;
        if ((r = ensure(J, J->nbulk, (size_t)4 * F * J->kb))) return r;
        if ((r = ensure(J, J->uk, (size_t)4 * F * J->K))) return r;
    }
    if (J->verify && J->atoms_family)
        if ((r = ensure(J, J->vrec, sizeof(VRec) * (size_t)F * NP * Mv))) return r;
    if (host_input) {
        if ((r = ensure(J, J->xin_u, (size_t)dtype_size * F * J->Nu * 3))) return r;
        if ((r = ensure(J, J->xin_v, (size_t)dtype_size * F * J->Nv * 3))) return r;
    }
    return CM_OK;
}

// the self-MDDF half range of the accumulators: both group hits of a record
// count w/2 (update_counters.jl:48-53)
void half_range(const cm_job* J, int64_t* lo, int64_t* hi)
{
    *lo = *hi = 0;
    if (J->d.autocorrelation) {
        *lo = 4 * (int64_t)J->d.nbins;
        *hi = J->acc_len;
    }
}

// assign: the hits of the job's first weight run go into accumulators that
// may hold anything (the packed read-back reuses their storage); with
// count_hits == false the md/rdf hits are not added to the cumulative ones
// (they already were)
int flush(cm_job* J, double w, hipStream_t stream = nullptr, bool assign = false, bool count_hits = true)
{
    int64_t nb = J->d.nbins;
    int64_t half_lo, half_hi;
    half_range(J, &half_lo, &half_hi);
    hipLaunchKernelGGL(k_flush, dim3(grid_for(J->acc_len)), dim3(BLOCK), 0, stream ? stream : J->stream, (ull*)J->cnt.p,
                       (double*)J->acc.p,
                       (ull*)J->hits.p, J->acc_len, count_hits ? 4 * nb : 0, half_lo, half_hi, w, assign ? 1 : 0);
    HIPCHK(hipGetLastError());
    J->flushes++;
    return CM_OK;
}

// cell slots per frame (the largest grid of the frames, with 10% headroom so
// that batches of later frames of a fluctuating box reuse the allocation) and
// frames per batch
int batch_plan(const cm_job* J, int32_t nframes, const double* cells, int ds, bool host_input, int64_t* capmax_,
               int64_t* kcapmax_, int64_t* Fmax_, int64_t* pfb_)
{
    int64_t capmax = 1, kcapmax = 1;
    for (int f = 0; f < nframes; f++) {
        int64_t kk;
        capmax = std::max(capmax, cells_for(J, cells + 9 * f, &kk));
        kcapmax = std::max(kcapmax, kk);
    }
    if (capmax > (int64_t)1 << 26 || kcapmax > (int64_t)1 << 27)
        return fail(CM_EUNSUPPORTED, "unit cell too large for the cell grid");
    capmax = capmax + capmax / 10 + 1;
    if (!J->atoms_family) kcapmax = 1;
    const int64_t pfb = per_frame_bytes(J, ds, host_input, capmax, kcapmax);
    const int64_t budget = J->d.memory_budget > 0 ? J->d.memory_budget : (int64_t)4 << 30;
    int64_t Fmax = std::max<int64_t>(1, budget / std::max<int64_t>(pfb, 1));
    if (J->d.max_batch_frames > 0) Fmax = std::min<int64_t>(Fmax, J->d.max_batch_frames);
    // at most 48 frames per batch: the random-pass evaluation of config-2 sized
    // jobs ran 25% slower per frame with 64-frame batches than with 32-48
    Fmax = std::min<int64_t>(Fmax, 48);
    *capmax_ = capmax;
    *kcapmax_ = kcapmax;
    *Fmax_ = Fmax;
    *pfb_ = pfb;
    return CM_OK;
}

int submit_common(cm_job* J, int32_t nframes, const int64_t* frame_index, const void* xu, const void* xv, int32_t dtype,
                  const double* cells, const double* weights, bool host_input)
{
    if (!J) return fail(CM_EINVAL, "null job");
    if (J->finished) return fail(CM_ESTATE, "job already finished");
    if (nframes < 0 || (nframes > 0 && (!frame_index || !xu || !xv || !cells || !weights)))
        return fail(CM_EINVAL, "invalid frame arrays");
    if (dtype != CM_F64 && dtype != CM_F32) return fail(CM_EINVAL, "dtype must be CM_F64 or CM_F32");
    int ds = dtype == CM_F32 ? 4 : 8;
    for (int f = 0; f < nframes; f++) {
        if (!(weights[f] > 0.0) || !std::isfinite(weights[f])) return fail(CM_EINVAL, "frame weights must be positive and finite");
        if (frame_index[f] < 1 || frame_index[f] > 0xFFFFFFFFll) return fail(CM_EINVAL, "frame_index must be in [1, 2^32)");
    }
    if (nframes == 0) return CM_OK;
    int64_t capmax, kcapmax, Fmax, pfb;
    int r0 = batch_plan(J, nframes, cells, ds, host_input, &capmax, &kcapmax, &Fmax, &pfb);
    if (r0) return r0;
    int f0 = 0;
    while (f0 < nframes) {
        // a batch holds frames of one weight (the weight multiplies the integer hits at flush)
        double w = weights[f0];
        // the frames of this weight in equal batches (200 frames: 5 x 40, not
        // 4 x 48 + 8)
        int run = 1;
        while (f0 + run < nframes && weights[f0 + run] == w) run++;
        const int nb = (int)((run + Fmax - 1) / Fmax);
        const int F = (run + nb - 1) / nb;
        if (J->pending && J->pending_w != w) {
            int r = flush(J, J->pending_w);
            if (r) return r;
        }
        J->pending = true;
        J->pending_w = w;
        const int64_t cap = capmax;
        for (int f = 0; f < F; f++) {
            cm::Cell64 c;
            cm::cell_setup(cells + 9 * (f0 + f), J->d.triclinic, &c);
            J->volume_total += w * cm::cell_volume(c.H);
        }
        int r = alloc_batch(J, F, cap, kcapmax, ds, host_input);
        if (r) return r;
        const void* du;
        const void* dv;
        if (host_input) {
            const void* su = (const char*)xu + (size_t)f0 * J->Nu * 3 * ds;
            const void* sv = (const char*)xv + (size_t)f0 * J->Nv * 3 * ds;
            HIPCHK(hipMemcpyAsync(J->xin_u.p, su, (size_t)F * J->Nu * 3 * ds, hipMemcpyHostToDevice, J->stream));
            HIPCHK(hipMemcpyAsync(J->xin_v.p, sv, (size_t)F * J->Nv * 3 * ds, hipMemcpyHostToDevice, J->stream));
            // Copies from pageable memory are staged before hipMemcpyAsync
            // returns; copies from page-locked memory run later, in stream
            // order.  The caller may reuse its arrays once the call returns,
            // so page-locked sources are waited for.
            if (page_locked(su) || page_locked(sv)) HIPCHK(hipStreamSynchronize(J->stream));
            du = J->xin_u.p;
            dv = J->xin_v.p;
        } else {
            du = (const char*)xu + (size_t)f0 * J->Nu * 3 * ds;
            dv = (const char*)xv + (size_t)f0 * J->Nv * 3 * ds;
        }
        r = run_batch(J, F, frame_index + f0, du, dv, dtype, cells + 9 * f0, cap, kcapmax);
        if (r) return r;
        f0 += F;
    }
    return CM_OK;
}

// argument checks of a job description (the messages the host maps to
// ArgumentError)
int validate_desc(const cm_job_desc& d)
{
    if (d.nmols_u < 1 || d.natoms_per_mol_u < 1 || d.nmols_v < 1 || d.natoms_per_mol_v < 1)
        return fail(CM_EINVAL, "selections must hold at least one molecule of at least one atom");
    if (d.irefatom < 1 || d.irefatom > d.natoms_per_mol_v)
        return fail(CM_EINVAL, "irefatom must be between 1 and natoms_per_mol_v");
    if (d.nbins < 1 || d.nbins > MAX_NBINS) return fail(CM_EINVAL, "nbins out of range [1, 8192]");
    if (!(d.binstep > 0.0) || !(d.cutoff > 0.0) || !(d.dbulk > 0.0)) return fail(CM_EINVAL, "binstep, cutoff and dbulk must be positive");
    if ((int64_t)cm::setbin(d.cutoff, d.binstep) != d.nbins) return fail(CM_EINVAL, "nbins must equal setbin(cutoff, binstep)");
    if (d.usecutoff ? !(d.dbulk < d.cutoff) : !(d.dbulk <= d.cutoff))
        return fail(CM_EINVAL, "dbulk must not exceed cutoff (the histogram range)");
    if (d.n_random_samples < 1 && !d.coordination_number_only) return fail(CM_EINVAL, "n_random_samples must be greater than 0");
    if (d.n_groups_u < 1 || d.n_groups_v < 1) return fail(CM_EINVAL, "group counts must be positive");
    if (!d.groups_u_ptr && d.n_groups_u != d.natoms_per_mol_u) return fail(CM_EINVAL, "n_groups_u must equal natoms_per_mol_u without custom groups");
    if (!d.groups_v_ptr && d.n_groups_v != (d.autocorrelation ? d.natoms_per_mol_u : d.natoms_per_mol_v))
        return fail(CM_EINVAL, "n_groups_v must equal the atoms per molecule without custom groups");
    if (d.autocorrelation && (d.nmols_u != d.nmols_v || d.natoms_per_mol_u != d.natoms_per_mol_v))
        return fail(CM_EINVAL, "autocorrelation needs identical solute and solvent selections");
    if (d.seed == 0) return fail(CM_EINVAL, "seed must be positive");
    int64_t Nu = (int64_t)d.nmols_u * d.natoms_per_mol_u, Nv = (int64_t)d.nmols_v * d.natoms_per_mol_v;
    if (Nu > INT32_MAX / 4 || Nv > INT32_MAX / 4) return fail(CM_EINVAL, "selections too large");
    if (d.groups_u_ptr) {
        if (!d.groups_u_idx) return fail(CM_EINVAL, "groups_u_idx missing");
        for (int64_t k = 0; k < d.groups_u_ptr[d.natoms_per_mol_u]; k++)
            if (d.groups_u_idx[k] < 0 || d.groups_u_idx[k] >= d.n_groups_u) return fail(CM_EINVAL, "solute group id out of range");
    }
    if (d.groups_v_ptr) {
        if (!d.groups_v_idx) return fail(CM_EINVAL, "groups_v_idx missing");
        const int64_t lim = d.autocorrelation ? d.n_groups_u : d.n_groups_v;
        for (int64_t k = 0; k < d.groups_v_ptr[Nv]; k++)
            if (d.groups_v_idx[k] < 0 || d.groups_v_idx[k] >= lim) return fail(CM_EINVAL, "solvent group id out of range");
    }
    return CM_OK;
}

// Molecules per chunk (one wavefront each) of the real pass: 64 / tile_c, or for
// molecules of other than three atoms what 64 / tile_c atoms make.  KM random
// passes place KM times the molecules in the same space, so their chunks hold
// up to four times as many in no more space (up to 128 atoms: eight tiles).
void set_chunks(cm_job* J)
{
    KP& P = J->kp;
    const int share = P.KM >= 8 ? 4 : (P.KM >= 3 ? 2 : 1);
    if (P.mol_lane) {
        P.mpt = 64 / J->tile_c;
        P.mpt_r = std::min(64, P.mpt * share);
    } else {
        const int at = 64 / J->tile_c, at_r = at * share;
        P.mpt = std::max(1, at / P.nv);
        P.mpt_r = std::max(1, std::min(64, at_r > 64 ? 2 * lane_molecules(P.nv) : at_r / P.nv));
        P.mpt_auto = J->tuned_c ? 0 : 1;
    }
}

// (re)initialises a job on its stream for a validated description; device
// buffers already held by J are kept and grown as needed
// host-side fields of a job for a validated description (no device work)
void job_params(cm_job* J, const cm_job_desc& d)
{
    const int64_t Nu = (int64_t)d.nmols_u * d.natoms_per_mol_u, Nv = (int64_t)d.nmols_v * d.natoms_per_mol_v;
    J->d = d;
    J->Nu = Nu;
    J->Nv = Nv;
    J->pending = false;
    J->pending_w = 0.0;
    J->flushes = 0;
    J->volume_total = 0.0;
    J->finished = false;
    J->profiling = false;
    J->eval_ms = J->total_ms = 0.0;
    J->eval_launches = J->total_launches = J->frames = 0;
    J->prof_used = J->prof_done = 0;
    J->verify = false;
    J->vstore.clear();
    J->prof_random.clear();
    J->launch_ms.clear();
    J->cell_frac = 0.5;
    J->eval_grid = 0;
    J->tuned_c = false;
    // tiles family: one solute molecule, solvent molecules that fit a wavefront
    J->atoms_family = (d.nmols_u == 1 && !d.autocorrelation && d.natoms_per_mol_v <= 64);
    J->K = d.coordination_number_only ? 0 : d.n_random_samples;
    J->kb = J->K > 0 ? (J->atoms_family ? 1 : J->K) : 0;
    KP& P = J->kp;
    memset(&P, 0, sizeof(P));
    P.Mu = d.nmols_u; P.nu = d.natoms_per_mol_u; P.Mv = d.nmols_v; P.nv = d.natoms_per_mol_v;
    P.self_ = d.autocorrelation ? 1 : 0;
    P.iref = d.irefatom - 1;
    P.nbins = d.nbins;
    P.usecutoff = d.usecutoff ? 1 : 0;
    P.binstep = d.binstep;
    P.cutsys = d.usecutoff ? d.cutoff : d.dbulk;
    P.cut2 = P.cutsys * P.cutsys;
    P.dbulk = d.dbulk;
    P.inv_binstep = (float)(1.0 / d.binstep);
    {
        auto down = [](double x) { float f = (float)x; return (double)f > x ? std::nextafter(f, -INFINITY) : f; };
        auto up = [](double x) { float f = (float)x; return (double)f < x ? std::nextafter(f, INFINITY) : f; };
        const double bs2 = d.binstep * d.binstep, db2 = d.dbulk * d.dbulk;
        P.c2lo32 = down(P.cut2);
        P.c2hi32 = up(P.cut2);
        P.bs2m32 = down(bs2 * (1.0 - 4e-7));
        P.bs2p32 = up(bs2 * (1.0 + 4e-7));
        P.db2lo32 = down(db2 * (1.0 - 4e-7));
        P.db2hi32 = up(db2 * (1.0 + 4e-7));
    }
    P.K = J->K;
    P.kb = J->kb;
    P.key0 = (uint32_t)d.seed;
    P.key1 = (uint32_t)(d.seed >> 32);
    P.Nu = Nu;
    P.Nv = Nv;
    P.NP = 1 + J->K;
    P.mol_lane = P.nv == 3 ? 1 : 0;
    // random passes merged into groups of at most 16 (and of fewer than 2^31
    // slots); eight or more passes per group get keys of half-cells
    {
        const int64_t most = std::max<int64_t>(1, std::min<int64_t>(16, (INT32_MAX - BLOCK) / std::max<int64_t>(P.Mv, 1)));
        P.NG = J->K > 0 ? (int)((J->K + most - 1) / most) : 0;
        P.KM = J->K > 0 ? (J->K + P.NG - 1) / P.NG : 1;
        P.NG = J->K > 0 ? (J->K + P.KM - 1) / P.KM : 0;
        P.ksub = J->K >= 8 * std::max(P.NG, 1) ? 1 : 0;
    }
    // Molecules a chunk of the real pass: 16 of one, two or three atoms, 8 and 6 of
    // four and five, beyond that 64 atoms.  Larger chunks stage solute atoms for
    // molecules they are not near (5,000 solute atoms, 8 frames, evaluation and
    // resolve: 12,600 single atoms 44 us with 16, 53 with 32, 78 with 64; 5,000
    // four-atom molecules 105 with 8, 118 with 16), smaller ones stage the same
    // atoms more often (6,500 eight-atom molecules 151 with 8, 177 with 4).
    J->tile_c = P.nv == 1 || P.mol_lane ? 4 : (P.nv <= 5 ? 2 : 1);
    set_chunks(J);
    // Molecule pairs on the matrix cores: molecules of up to CL_ATOMS atoms
    // on both sides, the rows of one tile.  Larger ones would need minima over
    // several tiles; their walk already spends its time on distances (one
    // thread, 289 of them or more a pair).  The no-allocation entry point keeps
    // the walk as well: tiles and clusters take more of its fixed scratch per frame
    // (three-atom molecules against themselves 165 to 180 bytes a molecule, the
    // walk 104), so jobs near its limit would be refused.
    if (!J->atoms_family && !J->arena && P.nu <= CL_ATOMS && P.nv <= CL_ATOMS) {
        P.rpm = P.nu == 1 && P.nv == 1 ? 1 : (P.nu <= 4 ? 4 : (P.nu <= 8 ? 8 : 16));
        P.nT = (int)(((int64_t)P.Mu * P.rpm + 15) / 16);
        P.nS = (P.nT + CL_SUP - 1) / CL_SUP;
        P.nB = (P.Mv + 15) / 16;
    }
    P.gnu = d.n_groups_u;
    P.gnv = d.n_groups_v;
    // molecule-pair kernels keep the group counts in LDS when they fit
    // (on the matrix cores the blocks are 16 wavefronts, one a CU, with 74 KB of
    // queues, so the groups may take more than in the walk's small blocks; out
    // of line, straight into the global counters, the groups of 14 + 3 atoms took
    // 118 of 312 us: 181 osmolytes in 16,667 waters, 20 frames)
    P.glds = (int64_t)d.nbins * (d.n_groups_u + (d.autocorrelation ? 0 : d.n_groups_v)) * 4 <= (P.rpm ? GLDS_MAX_CL : GLDS_MAX) ? 1 : 0;
    {
        int dev = 0;
        if (hipGetDevice(&dev) == hipSuccess)
            if (hipDeviceGetAttribute(&J->cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || J->cus < 1)
                J->cus = 256;
        J->lds_max = lds_per_block(dev);
    }
    J->acc_len = 4 * (int64_t)d.nbins + 2 * (int64_t)d.n_groups_u * d.nbins + 2 * (int64_t)d.n_groups_v * d.nbins;
}

int job_setup(cm_job* J, const cm_job_desc& d)
{
    job_params(J, d);
    KP& P = J->kp;
    const int64_t Nv = J->Nv;
    const int64_t nb = d.nbins;
    int r;
    if ((r = ensure(J, J->cnt, 8 * J->acc_len))) return r;
    if ((r = ensure(J, J->acc, 8 * J->acc_len))) return r;
    if ((r = ensure(J, J->hits, 8 * 4 * nb))) return r;
    if ((r = ensure(J, J->stats, 64))) return r;
    FillList fills;
    fills.add(J->cnt.p, 8 * J->acc_len);
    fills.add(J->acc.p, 8 * J->acc_len);
    fills.add(J->hits.p, 8 * 4 * nb);
    fills.add(J->stats.p, 64);
    if ((r = fill_async(fills, J->stream))) return r;
    // The page-locked read-back buffer is taken now, while the device is idle
    // for this job: page-locking tens of MB (hipHostMalloc) while the job's
    // kernels run stalled one of them about fourfold (a 2.4 ms evaluation took
    // 9.6 ms in the first job of a process, where the cache has no block yet).
    if (!J->arena) {
        const size_t need = 8 * (size_t)J->acc_len + 8 * 4 * (size_t)nb + 8;
        if (J->hres.bytes < need) {
            pin_put(J->hres);
            if ((r = pin_take(J->hres, need))) return r;
        }
    }
    // group maps
    std::vector<int32_t>& gm = J->hgm;
    gm.clear();
    int64_t ou_p = -1, ou_i = -1, ov_p = -1, ov_i = -1;
    if (d.groups_u_ptr) {
        const int64_t n = d.natoms_per_mol_u, m = d.groups_u_ptr[n];
        ou_p = gm.size(); gm.insert(gm.end(), d.groups_u_ptr, d.groups_u_ptr + n + 1);
        ou_i = gm.size(); gm.insert(gm.end(), d.groups_u_idx, d.groups_u_idx + m); gm.push_back(0);
    }
    if (d.groups_v_ptr) {
        const int64_t n = Nv, m = d.groups_v_ptr[n];
        ov_p = gm.size(); gm.insert(gm.end(), d.groups_v_ptr, d.groups_v_ptr + n + 1);
        ov_i = gm.size(); gm.insert(gm.end(), d.groups_v_idx, d.groups_v_idx + m); gm.push_back(0);
    }
    if (!gm.empty()) {
        if ((r = ensure(J, J->gmap, 4 * gm.size()))) return r;
        HIPCHK(hipMemcpyAsync(J->gmap.p, gm.data(), 4 * gm.size(), hipMemcpyHostToDevice, J->stream));
        HIPCHK(hipStreamSynchronize(J->stream));
        int32_t* base = (int32_t*)J->gmap.p;
        if (ou_p >= 0) { P.gu_ptr = base + ou_p; P.gu_idx = base + ou_i; }
        if (ov_p >= 0) { P.gv_ptr = base + ov_p; P.gv_idx = base + ov_i; }
    }
    J->d.groups_u_ptr = J->d.groups_u_idx = J->d.groups_v_ptr = J->d.groups_v_idx = nullptr;
    return CM_OK;
}

// The geometry error bits a job's batches left on the device (frame_grid):
// bit 0 molecules too large for the cell of the molecule-pair kernels, bit 1
// a cell grid larger than its allocation.  The same decoding for cm_job_finish
// and for the request server.
int geometry_error(uint64_t gerr)
{
    if (gerr & 1)
        return fail(CM_EUNSUPPORTED, "molecules too large for the unit cell: cutoff plus molecule radii exceed a plane spacing");
    if (gerr)
        return fail(CM_EHIP, "internal error: cell grid larger than its allocation");
    return CM_OK;
}

// Copies the read-back in h into the caller's arrays: FP64 accumulators, or
// 32-bit hits (packed) turned into (double)hits * w (w/2 in the self-MDDF
// group range), the product k_flush forms.  Worker threads take tasks of
// 256K entries; with ev, each first waits for the piece holding its task.
std::atomic<uint64_t>& pack_limit()
{
    static std::atomic<uint64_t> v{0xffffffffull};
    return v;
}

// Layout of a read-back in page-locked memory, for n accumulator entries of
// which the first nh = 4 nbins are the md/rdf histograms: the wire data
// (FP64 accumulators, or the 16-bit group counts of a packed read-back) in
// [0, 8 n), the cumulative md/rdf hits (64-bit), three flag words (geometry
// error bits, pack limit exceeded, number of overflowing counts), then the
// overflow list (entry, count) of a packed read-back.
struct RbLayout {
    int64_t n, nh, ng, ovcap;
    size_t off_hits, off_flags, off_ov, need, dev_ov;
    RbLayout(int64_t n_, int64_t nbins)
    {
        n = n_;
        nh = 4 * nbins;
        ng = n - nh;
        off_hits = 8 * (size_t)n;
        off_flags = off_hits + 8 * (size_t)nh;
        off_ov = off_flags + 32;
        // the overflow list sits in the accumulator block after the 16-bit words
        dev_ov = ((size_t)2 * ng + 15) & ~(size_t)15;
        ovcap = std::min<int64_t>(4096, (int64_t)((8 * (size_t)n - dev_ov) / 16));
        need = off_ov + 16 * (size_t)ovcap;
    }
};

// Writes a read-back (layout L in h) into the caller's arrays: FP64 copies,
// or for a packed read-back the products (double)count * w (w/2 in the
// self-MDDF group range [half_lo, half_hi)), the values k_flush forms; worker
// threads take tasks of 256K entries, and with ev each first waits for the
// wire piece holding its task.
int copy_out(const cm_job_desc& d, const RbLayout& L, const char* h, bool packed, double w, int64_t half_lo,
             int64_t half_hi, size_t piece, const hipEvent_t* ev, cm_raw* out)
{
    const int64_t nb = d.nbins, ngu = d.n_groups_u, ngv = d.n_groups_v;
    const int64_t n = L.n, nh = L.nh;
    const double wh = w / 2;
    auto mult = [&](int64_t k) { return (k >= half_lo && k < half_hi) ? wh : w; };
    // the caller's arrays as entry ranges of the accumulator block, in order
    struct Seg { int64_t o, n; double* dst; };
    std::vector<Seg> segs;
    int64_t o = 0;
    auto add = [&](double* dst, int64_t m) { if (dst && m) segs.push_back({o, m, dst}); o += m; };
    add(out->md_count, nb);
    add(out->md_count_random, nb);
    add(out->rdf_count, nb);
    add(out->rdf_count_random, nb);
    add(out->solute_group_count, ngu * nb);
    add(out->solvent_group_count, ngv * nb);
    add(out->solute_group_count_random, ngu * nb);
    add(out->solvent_group_count_random, ngv * nb);
    const ull* hits = (const ull*)(h + L.off_hits);
    const uint16_t* w16 = (const uint16_t*)h;
    constexpr int64_t TASK = (int64_t)1 << 18;
    const int64_t ntask = (n + TASK - 1) / TASK;
    hipError_t werr = hipSuccess;
    std::mutex werr_mu;
    auto work = [&](int64_t t0, int64_t step) {
        for (int64_t t = t0; t < ntask; t += step) {
            const int64_t a = t * TASK, b = std::min(n, a + TASK);
            if (ev) {
                // pieces land in stream order: the piece holding the task's last byte
                const size_t last = packed ? (b > nh ? 2 * (size_t)(b - 1 - nh) + 1 : 0) : 8 * (size_t)b - 1;
                if (!packed || b > nh) {
                    const hipError_t e = hipEventSynchronize(ev[last / piece]);
                    if (e != hipSuccess) {
                        std::lock_guard<std::mutex> lk(werr_mu);
                        werr = e;
                        return;
                    }
                }
            }
            for (const Seg& sg : segs) {
                const int64_t lo = std::max(a, sg.o), hi = std::min(b, sg.o + sg.n);
                if (lo >= hi) continue;
                double* dst = sg.dst + (lo - sg.o);
                if (!packed) {
                    memcpy(dst, h + 8 * lo, 8 * (size_t)(hi - lo));
                    continue;
                }
                // one multiplier per array (the self-MDDF half range is whole
                // arrays); signed conversions, a single instruction each
                const double m = mult(lo);
                if (hi <= nh) {
                    for (int64_t k = lo; k < hi; k++) dst[k - lo] = (double)(int64_t)hits[k] * m;
                } else {
                    const uint16_t* src = w16 + (lo - nh);
                    const int64_t cnt = hi - lo;
                    for (int64_t k = 0; k < cnt; k++) dst[k] = (double)(int32_t)src[k] * m;
                }
            }
        }
    };
    const int64_t nt = std::min<int64_t>(8, ntask);
    std::vector<std::thread> th;
    for (int64_t q = 1; q < nt; q++) th.emplace_back(work, q, nt);
    if (nt > 0) work(0, std::max<int64_t>(nt, 1));
    for (auto& x : th) x.join();
    if (werr != hipSuccess) return fail(CM_EHIP, std::string("read-back: ") + hipGetErrorString(werr));
    if (ev) HIPCHK(hipEventSynchronize(ev[RB_PIECES - 1]));
    if (packed) {
        // the counts that did not fit 16 bits
        uint64_t nov;
        memcpy(&nov, h + L.off_flags + 16, 8);
        const ulonglong2* ov = (const ulonglong2*)(h + L.off_ov);
        for (uint64_t q = 0; q < nov; q++) {
            const int64_t k = (int64_t)ov[q].x;
            for (const Seg& sg : segs)
                if (k >= sg.o && k < sg.o + sg.n) sg.dst[k - sg.o] = (double)ov[q].y * mult(k);
        }
    }
    auto cpu = [&](uint64_t* dst, const ull* src) { if (dst) memcpy(dst, src, 8 * nb); };
    cpu(out->hits_md, hits);
    cpu(out->hits_md_random, hits + nb);
    cpu(out->hits_rdf, hits + 2 * nb);
    cpu(out->hits_rdf_random, hits + 3 * nb);
    return CM_OK;
}

// The packed read-back of a one-weight job: k_pack16 into the accumulator
// block (its FP64 contents are not needed: the job has no flushed run)
void launch_pack16(cm_job* J, const RbLayout& L, hipStream_t s)
{
    hipLaunchKernelGGL(k_pack16, dim3(grid_for(L.n)), dim3(BLOCK), 0, s, (const ull*)J->cnt.p, (uint16_t*)J->acc.p,
                       (ull*)J->hits.p, L.n, L.nh, (ull)pack_limit().load(), (ull*)J->stats.p + 3,
                       (ulonglong2*)((char*)J->acc.p + L.dev_ov), L.ovcap);
}

// a packed read-back that cannot be decoded: a count above the pack limit,
// or more overflowing counts than the list holds
bool pack_failed(const RbLayout& L, const char* h)
{
    uint64_t fl[3];
    memcpy(fl, h + L.off_flags, 24);
    return fl[1] != 0 || fl[2] > (uint64_t)L.ovcap;
}

// Read-back of cm_job_finish, pipelined: the accumulators come back in
// RB_PIECES pieces, each with an event, and worker threads copy 256K-entry
// tasks into the caller's arrays as soon as the piece holding a task has
// landed, so the copies into (often freshly allocated, page-faulting) caller
// memory overlap the transfer.  The geometry error bits come back first.
//
// When every frame of the job had one weight w (no weight change flushed
// yet), each FP64 result is (double)hits * w (w/2 in the self-MDDF group
// range) with nothing added before it, so the group counts cross PCIe as
// 16-bit words (a quarter of the bytes of the accumulators; the few larger
// counts in a list beside them, the md/rdf histograms from the 64-bit hits)
// and the host forms the same products, rounded the same way.  A count above
// the pack limit, or more large counts than the list holds, sends the job
// down the FP64 path.
int job_finish_pipelined(cm_job* J, cm_raw* out)
{
    const cm_job_desc& d = J->d;
    const int64_t nb = d.nbins;
    const RbLayout L(J->acc_len, nb);
    hipStream_t s = J->stream;
    const bool packed = J->pending && J->flushes == 0;
    const double w = J->pending_w;
    if (packed) {
        launch_pack16(J, L, s);
        HIPCHK(hipGetLastError());
    } else if (J->pending) {
        if (int r = flush(J, J->pending_w)) return r;
    }
    J->pending = false;
    if (J->hres.bytes < L.need) {
        pin_put(J->hres);
        int r = pin_take(J->hres, L.need);
        if (r) return r;
    }
    for (auto& e : J->rb_ev)
        if (!e) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    char* h = (char*)J->hres.p;
    // error bits and the packing flags, the md/rdf hits, the overflow list
    HIPCHK(hipMemcpyAsync(h + L.off_flags, (char*)J->stats.p + 16, 24, hipMemcpyDeviceToHost, s));
    HIPCHK(hipMemcpyAsync(h + L.off_hits, J->hits.p, 8 * (size_t)L.nh, hipMemcpyDeviceToHost, s));
    if (packed)
        HIPCHK(hipMemcpyAsync(h + L.off_ov, (char*)J->acc.p + L.dev_ov, 16 * (size_t)L.ovcap, hipMemcpyDeviceToHost, s));
    HIPCHK(hipEventRecord(J->rb_ev[RB_PIECES], s));
    const size_t wire = packed ? 2 * (size_t)L.ng : 8 * (size_t)L.n;
    const size_t piece = ((wire + RB_PIECES - 1) / RB_PIECES + 4095) & ~(size_t)4095;
    for (int k = 0; k < RB_PIECES; k++) {
        const size_t o = std::min(wire, k * piece), m = std::min(wire, o + piece) - o;
        if (m) HIPCHK(hipMemcpyAsync(h + o, (char*)J->acc.p + o, m, hipMemcpyDeviceToHost, s));
        HIPCHK(hipEventRecord(J->rb_ev[k], s));
    }
    HIPCHK(hipEventSynchronize(J->rb_ev[RB_PIECES]));
    uint64_t gerr;
    memcpy(&gerr, h + L.off_flags, 8);
    if (int r = geometry_error(gerr)) return r;
    int64_t half_lo, half_hi;
    half_range(J, &half_lo, &half_hi);
    int r;
    if (packed && pack_failed(L, h)) {
        // the FP64 accumulators after all (the hits were already added to
        // the cumulative md/rdf ones)
        HIPCHK(hipStreamSynchronize(s));
        if ((r = flush(J, w, nullptr, true, false))) return r;
        HIPCHK(hipMemcpyAsync(h, J->acc.p, 8 * (size_t)L.n, hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        r = copy_out(d, L, h, false, w, half_lo, half_hi, piece, nullptr, out);
    } else {
        r = copy_out(d, L, h, packed, w, half_lo, half_hi, piece, J->rb_ev, out);
    }
    if (r) return r;
    out->volume_total = J->volume_total;
    J->finished = true;
    return CM_OK;
}

// Reads a finished request's results back into J->hres (layout RbLayout):
// the accumulators, or, when its frames shared one weight, the packed counts
// (*packed set, as in cm_job_finish), the md/rdf hits and the flags.
int job_collect(cm_job* J, bool* packed)
{
    const RbLayout L(J->acc_len, J->d.nbins);
    *packed = J->pending && J->flushes == 0;
    if (*packed) {
        launch_pack16(J, L, J->stream);
        HIPCHK(hipGetLastError());
    } else if (J->pending) {
        if (int r = flush(J, J->pending_w)) return r;
    }
    J->pending = false;
    if (J->hres.bytes < L.need) {
        pin_put(J->hres);
        int r = pin_take(J->hres, L.need);
        if (r) return r;
    }
    char* h = (char*)J->hres.p;
    HIPCHK(hipMemcpyAsync(h, J->acc.p, *packed ? 2 * (size_t)L.ng : 8 * (size_t)L.n, hipMemcpyDeviceToHost, J->stream));
    HIPCHK(hipMemcpyAsync(h + L.off_hits, J->hits.p, 8 * (size_t)L.nh, hipMemcpyDeviceToHost, J->stream));
    HIPCHK(hipMemcpyAsync(h + L.off_flags, (char*)J->stats.p + 16, 24, hipMemcpyDeviceToHost, J->stream));
    if (*packed)
        HIPCHK(hipMemcpyAsync(h + L.off_ov, (char*)J->acc.p + L.dev_ov, 16 * (size_t)L.ovcap, hipMemcpyDeviceToHost,
                              J->stream));
    HIPCHK(hipStreamSynchronize(J->stream));
    uint64_t gerr;
    memcpy(&gerr, h + L.off_flags, 8);
    if (int r = geometry_error(gerr)) return r;
    if (*packed && pack_failed(L, h)) {
        // FP64 accumulators (md/rdf hits already added)
        if (int r = flush(J, J->pending_w, nullptr, true, false)) return r;
        HIPCHK(hipMemcpyAsync(h, J->acc.p, 8 * (size_t)L.n, hipMemcpyDeviceToHost, J->stream));
        HIPCHK(hipStreamSynchronize(J->stream));
        *packed = false;
    }
    J->finished = true;
    return CM_OK;
}

// raw accumulators of a collected request into the caller's cm_raw
int fill_raw(const cm_job_desc& d, int64_t acc_len, const PinBuf& res, double volume, bool packed, double w,
             cm_raw* out)
{
    const RbLayout L(acc_len, d.nbins);
    const int64_t half_lo = d.autocorrelation ? L.nh : 0, half_hi = d.autocorrelation ? acc_len : 0;
    if (int r = copy_out(d, L, (const char*)res.p, packed, w, half_lo, half_hi, 1, nullptr, out)) return r;
    out->volume_total = volume;
    return CM_OK;
}

// Times of the batches profiled since the last call: waits for the job's
// stream, reads the event pairs and adds them to the job's totals.
int prof_resolve(cm_job* J)
{
    if (J->prof_done == J->prof_used) return CM_OK;
    HIPCHK(hipStreamSynchronize(J->stream));
    for (size_t b = J->prof_done; b < J->prof_used; b++) {
        const auto& e = J->prof_ev[b];
        const bool rnd = J->prof_random[b] != 0;
        float real = 0.f, ran = -1.f, tot = 0.f;
        HIPCHK(hipEventElapsedTime(&real, e[0], e[1]));
        if (rnd) HIPCHK(hipEventElapsedTime(&ran, e[2], e[3]));
        HIPCHK(hipEventElapsedTime(&tot, e[4], rnd ? e[3] : e[1]));
        J->eval_ms += real + (rnd ? ran : 0.f);
        J->eval_launches += rnd ? 2 : 1;
        J->total_ms += tot;
        J->total_launches += 1;
        J->launch_ms.emplace_back(real, ran);
    }
    J->prof_done = J->prof_used;
    return CM_OK;
}

}  // namespace

extern "C" {

const char* cm_last_error(void) { return g_err.c_str(); }

int cm_job_create(const cm_job_desc* desc, cm_job** out)
{
    if (!desc || !out) return fail(CM_EINVAL, "null argument");
    *out = nullptr;
    int r = validate_desc(*desc);
    if (r) return r;
    cm_job* J = new cm_job();
    if ((r = stream_take(&J->stream))) {
        cm_job_destroy(J);
        return r;
    }
    if ((r = job_setup(J, *desc))) {
        cm_job_destroy(J);
        return r;
    }
    *out = J;
    return CM_OK;
}

int cm_job_submit(cm_job* job, int32_t nframes, const int64_t* frame_index, const void* x_solute, const void* x_solvent,
                  int32_t dtype, const double* cells, const double* weights)
{
    return submit_common(job, nframes, frame_index, x_solute, x_solvent, dtype, cells, weights, true);
}

int cm_job_submit_device(cm_job* job, int32_t nframes, const int64_t* frame_index, const void* d_x_solute,
                         const void* d_x_solvent, int32_t dtype, const double* cells, const double* weights)
{
    return submit_common(job, nframes, frame_index, d_x_solute, d_x_solvent, dtype, cells, weights, false);
}

int cm_job_finish(cm_job* J, cm_raw* out)
{
    if (!J || !out) return fail(CM_EINVAL, "null argument");
    if (J->finished) return fail(CM_ESTATE, "job already finished");
    return job_finish_pipelined(J, out);
}

int cm_job_set_profiling(cm_job* J, int32_t on)
{
    if (!J) return fail(CM_EINVAL, "null job");
    J->profiling = on != 0;
    return CM_OK;
}

int cm_job_set_tuning(cm_job* J, double cell_fraction, int32_t columns, int32_t eval_workgroups)
{
    if (!J) return fail(CM_EINVAL, "null job");
    if (J->frames > 0) return fail(CM_ESTATE, "tuning must be set before the first submit");
    if (!(cell_fraction >= 0.2 && cell_fraction <= 1.0)) return fail(CM_EINVAL, "cell_fraction must be in [0.2, 1]");
    if (columns != 0 && columns != 1 && columns != 2 && columns != 4 && columns != 8)
        return fail(CM_EINVAL, "columns must be 0 (default), 1, 2, 4 or 8");
    const bool tuned = columns > 0;
    if (!tuned) columns = J->tile_c;
    if (!J->kp.mol_lane && (64 / columns) / J->kp.nv < 1) return fail(CM_EINVAL, "too many columns for the solvent molecule size");
    if (eval_workgroups < 0) return fail(CM_EINVAL, "eval_workgroups must be >= 0");
    J->cell_frac = cell_fraction;
    J->tuned_c = tuned;
    J->tile_c = columns;
    set_chunks(J);
    J->eval_grid = eval_workgroups;
    return CM_OK;
}

int cm_job_kernel_stats(cm_job* J, cm_kernel_stats* out)
{
    if (!J || !out) return fail(CM_EINVAL, "null argument");
    if (int r = prof_resolve(J)) return r;
    ull st[2] = {0, 0};
    HIPCHK(hipMemcpyAsync(st, J->stats.p, 16, hipMemcpyDeviceToHost, J->stream));
    HIPCHK(hipStreamSynchronize(J->stream));
    out->eval_ms = J->eval_ms;
    out->eval_launches = J->eval_launches;
    out->total_ms = J->total_ms;
    out->total_launches = J->total_launches;
    out->frames = J->frames;
    out->candidate_pairs = -1;
    out->fp64_rechecks = (int64_t)st[0];
    return CM_OK;
}

int cm_job_launch_times(cm_job* J, int32_t cap, double* real_ms, double* random_ms, int32_t* n)
{
    if (!J || !n || (cap > 0 && (!real_ms || !random_ms))) return fail(CM_EINVAL, "null argument");
    if (int r = prof_resolve(J)) return r;
    *n = (int32_t)J->launch_ms.size();
    for (int32_t k = 0; k < cap && k < *n; k++) {
        real_ms[k] = J->launch_ms[k].first;
        random_ms[k] = J->launch_ms[k].second;
    }
    return CM_OK;
}

int cm_job_set_verify(cm_job* J, int32_t on)
{
    if (!J) return fail(CM_EINVAL, "null job");
    if (J->frames > 0) return fail(CM_ESTATE, "verification must be set before the first submit");
    if (J->arena) return fail(CM_EUNSUPPORTED, "no verification on the no-allocation path");
    J->verify = on != 0;
    J->kp.place_all = J->verify ? 1 : 0;
    return CM_OK;
}

int cm_job_records(cm_job* J, int64_t frame, int32_t pass, cm_md_record* out)
{
    if (!J || !out) return fail(CM_EINVAL, "null argument");
    if (!J->verify) return fail(CM_ESTATE, "verification is off for this job");
    if (!J->atoms_family)
        return fail(CM_EUNSUPPORTED, "records are kept for jobs with one solute molecule (tile kernels) only");
    if (pass < 0 || pass > J->K) return fail(CM_EINVAL, "pass must be 0 (real) or 1..n_random_samples");
    auto it = J->vstore.find(frame);
    if (it == J->vstore.end()) return fail(CM_EINVAL, "frame not processed by this job");
    static_assert(sizeof(VRec) == sizeof(cm_md_record), "record layout");
    std::memcpy(out, it->second.rec.data() + (size_t)pass * J->d.nmols_v, sizeof(VRec) * (size_t)J->d.nmols_v);
    return CM_OK;
}

int cm_job_placement(cm_job* J, int64_t frame, int32_t pass, double* out, uint8_t* placed)
{
    if (!J || !out || !placed) return fail(CM_EINVAL, "null argument");
    if (!J->verify) return fail(CM_ESTATE, "verification is off for this job");
    if (pass < 1 || pass > J->K) return fail(CM_EINVAL, "pass must be 1..n_random_samples");
    auto it = J->vstore.find(frame);
    if (it == J->vstore.end()) return fail(CM_EINVAL, "frame not processed by this job");
    const int64_t k = pass - 1;
    std::memcpy(out, it->second.placed.data() + (size_t)k * J->Nv * 3, sizeof(double) * 3 * (size_t)J->Nv);
    std::memcpy(placed, it->second.placed_flag.data() + (size_t)k * J->d.nmols_v, (size_t)J->d.nmols_v);
    return CM_OK;
}

int cm_job_reference_draws(cm_job* J, int64_t frame, int32_t* out)
{
    if (!J || !out) return fail(CM_EINVAL, "null argument");
    if (!J->verify) return fail(CM_ESTATE, "verification is off for this job");
    auto it = J->vstore.find(frame);
    if (it == J->vstore.end()) return fail(CM_EINVAL, "frame not processed by this job");
    std::memcpy(out, it->second.draws.data(), sizeof(int32_t) * (size_t)J->K);
    return CM_OK;
}

void cm_job_destroy(cm_job* J)
{
    if (!J) return;
    if (J->stream) (void)hipStreamSynchronize(J->stream);
    DevBuf* bufs[] = {&J->cnt, &J->acc, &J->hits, &J->stats, &J->gmap, &J->geo, &J->cells_cnt, &J->cells_start,
                      &J->tmp4, &J->tmpcell, &J->sorted, &J->solw, &J->ucen, &J->vw, &J->vcell, &J->vcen, &J->P,
                      &J->vw_r, &J->vcen_r, &J->bflag, &J->blist, &J->nbulk, &J->uk, &J->drawn_ptr,
                      &J->drawn_idx, &J->xin_u, &J->xin_v, &J->near, &J->mkey, &J->mrank, &J->mcnt, &J->mstart, &J->msum,
                      &J->clmem, &J->msorted, &J->nnear, &J->chunk_base, &J->vrec};
    for (DevBuf* b : bufs) dev_put(*b);
    pin_put(J->hres);
    for (auto& a : J->prof_ev)
        for (auto& e : a) (void)hipEventDestroy(e);
    for (auto& e : J->rb_ev)
        if (e) (void)hipEventDestroy(e);
    stream_put(J->stream);
    delete J;
}

int cm_set_readback_pack_limit(uint64_t limit)
{
    if (limit > 0xffffffffull) return fail(CM_EINVAL, "the pack limit is at most 2^32 - 1");
    pack_limit().store(limit);
    return CM_OK;
}

int cm_release_cached_memory(void)
{
    for (auto& blk : cache_drain(dev_cache())) HIPCHK(hipFree(blk.second));
    for (auto& blk : cache_drain(pin_cache())) HIPCHK(hipHostFree(blk.second));
    return CM_OK;
}

int cm_device_alloc(size_t bytes, void** dptr)
{
    if (!dptr) return fail(CM_EINVAL, "null pointer");
    hipError_t e = hipMalloc(dptr, bytes ? bytes : 16);
    if (e != hipSuccess) return fail(CM_ENOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    return CM_OK;
}

int cm_device_upload(void* dptr, const void* host, size_t bytes)
{
    HIPCHK(hipMemcpy(dptr, host, bytes, hipMemcpyHostToDevice));
    return CM_OK;
}

int cm_device_free(void* dptr)
{
    HIPCHK(hipFree(dptr));
    return CM_OK;
}

int cm_device_synchronize(void)
{
    HIPCHK(hipDeviceSynchronize());
    return CM_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// request server: slots (one stream and one pooled job each) take requests in
// arrival order when the footprint estimates of the admitted ones fit the budget
// ---------------------------------------------------------------------------
namespace {

struct SrvReq {
    uint64_t id = 0;
    cm_job_desc d{};
    std::vector<int32_t> gup, gui, gvp, gvi;
    std::vector<int64_t> fi;
    std::vector<double> cells, w;
    const void* xu = nullptr;
    const void* xv = nullptr;
    int32_t nframes = 0, dtype = 0;
    double cf = 0.0;
    int32_t cols = 0;
    int64_t foot = 0;
    bool done = false;
    bool waited = false;             // a cm_server_wait has taken the ticket
    int status = CM_OK;
    std::string err;
    PinBuf res;                     // read-back accumulators (taken over from the slot's job)
    int64_t acc_len = 0;
    bool packed = false;            // res holds 32-bit hits of frames of weight wt
    double wt = 0.0;
    double volume = 0.0;
    cm_request_times t{};
    ~SrvReq() { pin_put(res); }
};

int64_t job_footprint(const cm_job_desc& d, int32_t nframes, int32_t dtype, const double* cells, int64_t* bytes)
{
    cm_job J;
    job_params(&J, d);
    int64_t cap, kcap, Fmax, pfb;
    int r = batch_plan(&J, nframes, cells, dtype == CM_F32 ? 4 : 8, false, &cap, &kcap, &Fmax, &pfb);
    if (r) return r;
    int64_t groups = 0;
    if (d.groups_u_ptr) groups += 4 * ((int64_t)d.natoms_per_mol_u + 2 + d.groups_u_ptr[d.natoms_per_mol_u]);
    if (d.groups_v_ptr) groups += 4 * (J.Nv + 2 + d.groups_v_ptr[J.Nv]);
    *bytes = 16 * J.acc_len + 32 * (int64_t)d.nbins + 64 + groups + std::min<int64_t>(Fmax, nframes) * pfb;
    return CM_OK;
}

}  // namespace

struct cm_server {
    int slots = 4;
    int64_t budget = 0;
    int device = 0;
    std::mutex m;
    std::condition_variable cv_work, cv_done;
    std::deque<SrvReq*> queue;
    std::unordered_map<uint64_t, SrvReq*> reqs;
    int64_t reserved = 0;
    bool stop = false;
    uint64_t next = 1;
    std::vector<cm_job*> shells;
    std::vector<std::thread> workers;
    std::chrono::steady_clock::time_point t0;
    double now() const { return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count(); }
};

namespace {

int run_request(cm_job* J, SrvReq* q)
{
    cm_job_desc d = q->d;
    d.groups_u_ptr = q->gup.empty() ? nullptr : q->gup.data();
    d.groups_u_idx = q->gup.empty() ? nullptr : q->gui.data();
    d.groups_v_ptr = q->gvp.empty() ? nullptr : q->gvp.data();
    d.groups_v_idx = q->gvp.empty() ? nullptr : q->gvi.data();
    int r = job_setup(J, d);
    if (r) return r;
    if (q->cf > 0.0 || q->cols > 0)
        if ((r = cm_job_set_tuning(J, q->cf > 0.0 ? q->cf : 0.5, q->cols, 0))) return r;
    if ((r = submit_common(J, q->nframes, q->fi.data(), q->xu, q->xv, q->dtype, q->cells.data(), q->w.data(), false)))
        return r;
    const double w = J->pending_w;
    bool packed = false;
    if ((r = job_collect(J, &packed))) return r;
    q->packed = packed;
    q->wt = w;
    q->res = J->hres;
    J->hres = PinBuf{};
    q->acc_len = J->acc_len;
    q->volume = J->volume_total;
    return CM_OK;
}

void serve_slot(cm_server* S, int k)
{
    // the device current when the server was created (hipGetDevice returned it)
    (void)hipSetDevice(S->device);
    cm_job* J = S->shells[k];
    for (;;) {
        SrvReq* q;
        {
            std::unique_lock<std::mutex> lk(S->m);
            S->cv_work.wait(lk, [&] {
                if (S->queue.empty()) return S->stop;
                // arrival order; a request larger than the budget runs alone
                return S->reserved == 0 || S->reserved + S->queue.front()->foot <= S->budget;
            });
            if (S->queue.empty()) return;
            q = S->queue.front();
            S->queue.pop_front();
            S->reserved += q->foot;
            q->t.started = S->now();
        }
        const int r = run_request(J, q);
        {
            std::lock_guard<std::mutex> lk(S->m);
            S->reserved -= q->foot;
            q->status = r;
            if (r) q->err = g_err;
            q->t.finished = S->now();
            q->done = true;
        }
        S->cv_done.notify_all();
        S->cv_work.notify_all();
    }
}

}  // namespace

extern "C" {

int cm_job_footprint(const cm_job_desc* desc, int32_t nframes, int32_t dtype, const double* cells, int64_t* bytes)
{
    if (!desc || !bytes || (nframes > 0 && !cells)) return fail(CM_EINVAL, "null argument");
    if (nframes < 0) return fail(CM_EINVAL, "nframes must be >= 0");
    if (dtype != CM_F64 && dtype != CM_F32) return fail(CM_EINVAL, "dtype must be CM_F64 or CM_F32");
    int r = validate_desc(*desc);
    if (r) return r;
    return (int)job_footprint(*desc, nframes, dtype, cells, bytes);
}

int cm_server_create(const cm_server_desc* desc, cm_server** out)
{
    if (!out) return fail(CM_EINVAL, "null argument");
    *out = nullptr;
    const int slots = desc && desc->slots > 0 ? desc->slots : 4;
    if (slots > 64) return fail(CM_EINVAL, "at most 64 slots");
    cm_server* S = new cm_server();
    S->slots = slots;
    S->budget = desc && desc->memory_budget > 0 ? desc->memory_budget : (int64_t)200 << 30;
    S->t0 = std::chrono::steady_clock::now();
    if (hipGetDevice(&S->device) != hipSuccess) {
        delete S;
        return fail(CM_EHIP, "hipGetDevice failed");
    }
    for (int k = 0; k < slots; k++) {
        cm_job* J = new cm_job();
        if (hipStreamCreateWithFlags(&J->stream, hipStreamNonBlocking) != hipSuccess) {
            cm_job_destroy(J);
            cm_server_destroy(S);
            return fail(CM_EHIP, "hipStreamCreate failed");
        }
        S->shells.push_back(J);
    }
    for (int k = 0; k < slots; k++) S->workers.emplace_back(serve_slot, S, k);
    *out = S;
    return CM_OK;
}

int cm_server_enqueue(cm_server* S, const cm_request* req, uint64_t* ticket)
{
    if (!S || !req || !req->job || !ticket) return fail(CM_EINVAL, "null argument");
    const cm_job_desc& d = *req->job;
    int r = validate_desc(d);
    if (r) return r;
    if (req->nframes < 1 || !req->frame_index || !req->d_x_solute || !req->d_x_solvent || !req->cells || !req->weights)
        return fail(CM_EINVAL, "invalid frame arrays");
    if (req->dtype != CM_F64 && req->dtype != CM_F32) return fail(CM_EINVAL, "dtype must be CM_F64 or CM_F32");
    for (int f = 0; f < req->nframes; f++) {
        if (!(req->weights[f] > 0.0) || !std::isfinite(req->weights[f])) return fail(CM_EINVAL, "frame weights must be positive and finite");
        if (req->frame_index[f] < 1 || req->frame_index[f] > 0xFFFFFFFFll) return fail(CM_EINVAL, "frame_index must be in [1, 2^32)");
    }
    if (req->cell_fraction != 0.0 && !(req->cell_fraction >= 0.2 && req->cell_fraction <= 1.0))
        return fail(CM_EINVAL, "cell_fraction must be in [0.2, 1]");
    if (req->columns != 0 && req->columns != 1 && req->columns != 2 && req->columns != 4 && req->columns != 8)
        return fail(CM_EINVAL, "columns must be 0 (default), 1, 2, 4 or 8");
    SrvReq* q = new SrvReq();
    q->d = d;
    const int64_t Nv = (int64_t)d.nmols_v * d.natoms_per_mol_v;
    if (d.groups_u_ptr) {
        q->gup.assign(d.groups_u_ptr, d.groups_u_ptr + d.natoms_per_mol_u + 1);
        q->gui.assign(d.groups_u_idx, d.groups_u_idx + d.groups_u_ptr[d.natoms_per_mol_u]);
    }
    if (d.groups_v_ptr) {
        q->gvp.assign(d.groups_v_ptr, d.groups_v_ptr + Nv + 1);
        q->gvi.assign(d.groups_v_idx, d.groups_v_idx + d.groups_v_ptr[Nv]);
    }
    q->d.groups_u_ptr = q->d.groups_u_idx = q->d.groups_v_ptr = q->d.groups_v_idx = nullptr;
    q->fi.assign(req->frame_index, req->frame_index + req->nframes);
    q->cells.assign(req->cells, req->cells + 9 * (size_t)req->nframes);
    q->w.assign(req->weights, req->weights + req->nframes);
    q->xu = req->d_x_solute;
    q->xv = req->d_x_solvent;
    q->nframes = req->nframes;
    q->dtype = req->dtype;
    q->cf = req->cell_fraction;
    q->cols = req->columns;
    if ((r = (int)job_footprint(d, req->nframes, req->dtype, req->cells, &q->foot))) {
        delete q;
        return r;
    }
    {
        std::lock_guard<std::mutex> lk(S->m);
        if (S->stop) {
            delete q;
            return fail(CM_ESTATE, "server is shutting down");
        }
        q->id = S->next++;
        q->t.enqueued = S->now();
        S->reqs[q->id] = q;
        S->queue.push_back(q);
        *ticket = q->id;
    }
    S->cv_work.notify_all();
    return CM_OK;
}

int cm_server_wait(cm_server* S, uint64_t ticket, cm_raw* out, cm_request_times* times)
{
    if (!S) return fail(CM_EINVAL, "null server");
    SrvReq* q;
    {
        std::unique_lock<std::mutex> lk(S->m);
        auto it = S->reqs.find(ticket);
        if (it == S->reqs.end() || it->second->waited) return fail(CM_EINVAL, "unknown ticket");
        q = it->second;
        // a second waiter on the same ticket is refused while this one waits
        q->waited = true;
        // the map may rehash while the lock is released inside wait (an
        // enqueue on another thread inserts): the entry is erased by key
        S->cv_done.wait(lk, [&] { return q->done; });
        S->reqs.erase(ticket);
    }
    if (times) *times = q->t;
    int st = q->status;
    if (st == CM_OK) {
        if (out) st = fill_raw(q->d, q->acc_len, q->res, q->volume, q->packed, q->wt, out);
    } else {
        g_err = q->err;
    }
    delete q;
    return st;
}

void cm_server_destroy(cm_server* S)
{
    if (!S) return;
    {
        std::lock_guard<std::mutex> lk(S->m);
        S->stop = true;
    }
    S->cv_work.notify_all();
    for (auto& t : S->workers) t.join();
    for (cm_job* J : S->shells) cm_job_destroy(J);
    for (auto& kv : S->reqs) delete kv.second;
    delete S;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// many jobs per round (cm_jobs_submit_device)
// ---------------------------------------------------------------------------
namespace {

constexpr int MR_MAX_DEVICES = 64;
constexpr int MS_FMAX = 48;        // frames of one job per round (the single-job batch cap)
// Blocks of the stage launches.  The slot stages have one virtual block per
// (256 slots, frame, pass) of every job, most of which exit at once (their
// slots are not near); a block walks its virtual blocks one after another,
// so the grids are large enough that each walks a few dozen at most (a grid
// of 2048 took 1.8x the single-job launches' time in the near placement).
constexpr int MG_256 = 32768;      // blocks of the 256-thread stage launches
constexpr int MG_1024 = 4096;      // blocks of the 1024-thread stage launches
constexpr int MG_RES = 4096;       // blocks of the resolve launches
constexpr int64_t MULTI_BUDGET = (int64_t)64 << 30;   // batch buffers of one submission's jobs together

struct MultiRunner {
    std::mutex m;
    bool ready = false;
    hipStream_t stream = nullptr;
    void* tab = nullptr;                  // device table and geometry area (fixed address: graphs use it)
    size_t tab_bytes = 0;
    void* htab[2] = {nullptr, nullptr};   // page-locked staging of the table, used in turn
    hipEvent_t up[2] = {nullptr, nullptr};
    int cur = 0;
    bool graphs = true;
    std::map<int, hipGraphExec_t> exec;   // per kernel variant
    hipEvent_t done = nullptr;
    int cus = 256;
    int64_t rounds = 0, launches = 0;
};

MultiRunner* multi_runners()
{
    static MultiRunner* r = new MultiRunner[MR_MAX_DEVICES];
    return r;
}

// upload layout: the table, the two evaluation launches' chunk counters
// (zero in every upload), the frames' Geo records
constexpr size_t MT_CTR_OFF = (sizeof(MultiTab) + 255) & ~(size_t)255;
constexpr size_t MT_GEO_OFF = MT_CTR_OFF + 256;

int multi_init(MultiRunner& R)
{
    if (R.ready) return CM_OK;
    HIPCHK(hipStreamCreateWithFlags(&R.stream, hipStreamNonBlocking));
    R.tab_bytes = MT_GEO_OFF + sizeof(Geo) * (size_t)MS_MAX * MS_FMAX;
    HIPCHK(hipMalloc(&R.tab, R.tab_bytes));
    for (int k = 0; k < 2; k++) {
        HIPCHK(hipHostMalloc(&R.htab[k], R.tab_bytes, hipHostMallocDefault));
        HIPCHK(hipEventCreateWithFlags(&R.up[k], hipEventDisableTiming));
    }
    HIPCHK(hipEventCreateWithFlags(&R.done, hipEventDisableTiming));
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess)
        if (hipDeviceGetAttribute(&R.cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || R.cus < 1) R.cus = 256;
    R.ready = true;
    return CM_OK;
}

template <class KERN>
int persistent_grid(KERN kern, int threads, size_t shm, int cus)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, threads, shm) != hipSuccess || nb < 1) nb = 1;
    return nb * cus;
}

// LDS words of the histograms of a group of jobs (their largest): part of the
// kernel variant, as the launches' LDS is fixed when a round is captured
int multi_hist_words(const KP& P)
{
    const int w = (EvHist::words(P) + 3) & ~3;
    return (w + 1023) / 1024 * 1024;
}

// the stage launches of one round (every argument but the table address is
// fixed per kernel variant, so the sequence can be captured and replayed)
// (g, gr: chunk_groups of its jobs)
template <class T, int TQ, bool RANDOM>
auto multi_eval(int g) -> void (*)(const MultiTab*, int*)
{
    if constexpr (TQ == ATOMS) return g == 8 ? km_eval_tiles<T, T, RANDOM, 8, TQ> : km_eval_tiles<T, T, RANDOM, 4, TQ>;
    else return g == 4 ? km_eval_tiles<T, T, RANDOM, 4, TQ> : (g == 2 ? km_eval_tiles<T, T, RANDOM, 2, TQ> : km_eval_tiles<T, T, RANDOM, 1, TQ>);
}

template <class T, int TQ>
void multi_launch(int g, int gr, hipStream_t s, const MultiTab* tab, int hist, int lds_max, int cus)
{
    auto ev_real = multi_eval<T, TQ, false>(g);
    auto ev_rand = multi_eval<T, TQ, true>(gr);
    // (the chunk tables of multi_tickets are static LDS)
    auto waves = [&](int n) {
        return (int)std::max<int64_t>(1, std::min<int64_t>(16, (lds_max - 2048 - 4 * (int64_t)hist) / (4 * (int64_t)eval_wave_words(n, TQ))));
    };
    const int w_real = waves(g), w_rand = waves(gr);
    const size_t shm = 4 * ((size_t)hist + (size_t)w_real * eval_wave_words(g, TQ));
    const size_t shm_r = 4 * ((size_t)hist + (size_t)w_rand * eval_wave_words(gr, TQ));
    // persistent grids of the two evaluations
    const int g_real = persistent_grid(ev_real, 64 * w_real, shm, cus);
    const int g_rand = persistent_grid(ev_rand, 64 * w_rand, shm_r, cus);
    hipLaunchKernelGGL(km_zero, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_radii<T>, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_wrap_atoms<T>, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_scan_cells, dim3(MG_1024), dim3(1024), 0, s, tab);
    hipLaunchKernelGGL(km_scatter, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_near_mark, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_dfield, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_bulk_init, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_prep_solvent_tiles<T>, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_scan_sums<false>, dim3(MG_1024), dim3(1024), 0, s, tab);
    hipLaunchKernelGGL(km_scan_rows<false>, dim3(MG_1024), dim3(1024), 0, s, tab);
    hipLaunchKernelGGL(km_mol_scatter<false>, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_fill_real<T>, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_chunk_table<false>, dim3(MG_1024), dim3(1024), 0, s, tab);
    int* ctr = (int*)((char*)tab + MT_CTR_OFF);
    hipLaunchKernelGGL(ev_real, dim3(g_real), dim3(64 * w_real), shm, s, tab, ctr);
    hipLaunchKernelGGL((km_resolve<T, T, false>), dim3(MG_RES), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_bulk_compact, dim3(MG_1024), dim3(1024), 0, s, tab);
    hipLaunchKernelGGL(km_place_keys, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_scan_sums<true>, dim3(MG_1024), dim3(1024), 0, s, tab);
    hipLaunchKernelGGL(km_scan_rows<true>, dim3(MG_1024), dim3(1024), 0, s, tab);
    hipLaunchKernelGGL(km_mol_scatter<true>, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_place_near<T>, dim3(MG_256), dim3(BLOCK), 0, s, tab);
    hipLaunchKernelGGL(km_chunk_table<true>, dim3(MG_1024), dim3(1024), 0, s, tab);
    hipLaunchKernelGGL(ev_rand, dim3(g_rand), dim3(64 * w_rand), shm_r, s, tab, ctr + 1);
    hipLaunchKernelGGL((km_resolve<T, T, true>), dim3(MG_RES), dim3(BLOCK), 0, s, tab);
}

void multi_launch_any(int dtype, const cm_job* J, hipStream_t s, const MultiTab* tab, int cus)
{
    const int g = chunk_groups(J->kp, false), gr = chunk_groups(J->kp, true);
    const int hist = multi_hist_words(J->kp), lds_max = J->lds_max;
    if (dtype == CM_F32) {
        if (J->kp.mol_lane) multi_launch<float, 3>(g, gr, s, tab, hist, lds_max, cus);
        else multi_launch<float, ATOMS>(g, gr, s, tab, hist, lds_max, cus);
    } else {
        if (J->kp.mol_lane) multi_launch<double, 3>(g, gr, s, tab, hist, lds_max, cus);
        else multi_launch<double, ATOMS>(g, gr, s, tab, hist, lds_max, cus);
    }
}

// jobs that share the kernels of a round's launches
int multi_variant(int dtype, const cm_job* J)
{
    return (dtype == CM_F32 ? 1 : 0) | (J->kp.mol_lane ? 2 : 0) | (chunk_groups(J->kp, false) << 2) |
           (chunk_groups(J->kp, true) << 6) | (multi_hist_words(J->kp) << 10);
}

// one job's part of a multi-job submission
struct MJob {
    cm_job* J = nullptr;
    const cm_frames* fr = nullptr;
    int64_t cap = 0, kcap = 0;
    std::vector<std::pair<int, int>> batches;   // (first frame, frames)
};

// blocks of each stage's grid for one job's batch of F frames, as the
// single-job launches size them: (x extent, total)
void stage_blocks(const KP& P, int F, const int64_t z16[3], int nbx[MS_N], int cnt[MS_N])
{
    auto set = [&](int st, int64_t x, int64_t y) {
        x = std::max<int64_t>(x, 1);
        nbx[st] = (int)x;
        cnt[st] = (int)(x * std::max<int64_t>(y, 0));
    };
    const int64_t mvb = (P.Mv + BLOCK - 1) / BLOCK;
    const int K = P.K;
    set(MS_ZERO, std::min<int64_t>(1024, std::max<int64_t>(1, (z16[0] + z16[1] + z16[2] + BLOCK - 1) / BLOCK)), 1);
    set(MS_RADII, std::min<int64_t>(mvb, 64), F);
    set(MS_WRAP, grid_for((int64_t)F * P.nu), 1);
    set(MS_SCAN_CELLS, F, 1);
    set(MS_SCATTER, grid_for((int64_t)F * P.nu), 1);
    set(MS_NEAR, near_blocks(P.nu), std::min(F, 65535));
    set(MS_DFIELD, grid_for((int64_t)F * P.cap * 16), 1);
    set(MS_PREP, grid_for((int64_t)F * P.Mv), 1);
    const int p0 = scan_parts(P.kcap), pk = scan_parts(P.kcapr);
    set(MS_SCAN_SUMS0, p0, p0 > 1 ? F : 0);
    set(MS_SCAN_ROWS0, p0, F);
    set(MS_MOL_SCATTER0, mvb, std::min(F, 65535));
    set(MS_FILL, grid_for((int64_t)F * P.Mv), 1);
    set(MS_CHUNK0, 1, 1);
    set(MS_BULK_INIT, grid_for((int64_t)F * P.kb * P.Mv), K > 0 ? 1 : 0);
    set(MS_BULK_COMPACT, (int64_t)F * P.kb, K > 0 ? 1 : 0);
    set(MS_PLACE_KEYS, mvb, K > 0 ? std::min(F * K, 65535) : 0);
    set(MS_SCAN_SUMSK, pk, K > 0 && pk > 1 ? F * P.NG : 0);
    set(MS_SCAN_ROWSK, pk, K > 0 ? F * P.NG : 0);
    const int64_t gvb = ((int64_t)P.KM * P.Mv + BLOCK - 1) / BLOCK;
    set(MS_MOL_SCATTERK, gvb, K > 0 ? std::min(F * P.NG, 65535) : 0);
    set(MS_PLACE_NEAR, gvb, K > 0 ? std::min(F * P.NG, 65535) : 0);
    set(MS_CHUNKK, 1, K > 0 ? 1 : 0);
    set(MS_RESOLVE0, resolve_parts(P, false), F);
    set(MS_RESOLVEK, K > 0 ? resolve_parts(P, true) : 1, K > 0 ? F * P.NG : 0);
}

// the rounds of one group of jobs that share the kernel variant
int multi_run_group(MultiRunner& R, std::vector<MJob>& grp, int dtype)
{
    const int ds = dtype == CM_F32 ? 4 : 8;
    const cm_job* J0 = grp[0].J;
    const int variant = multi_variant(dtype, J0);
    size_t maxr = 0;
    for (auto& m : grp) maxr = std::max(maxr, m.batches.size());
    for (size_t r = 0; r < maxr; r++) {
        std::vector<MJob*> act;
        for (auto& m : grp)
            if (r < m.batches.size()) act.push_back(&m);
        for (size_t a0 = 0; a0 < act.size(); a0 += MS_MAX) {
            const int n = (int)std::min<size_t>(MS_MAX, act.size() - a0);
            // the staging buffer's previous upload must have been read
            HIPCHK(hipEventSynchronize(R.up[R.cur]));
            MultiTab* T = (MultiTab*)R.htab[R.cur];
            Geo* gh = (Geo*)((char*)R.htab[R.cur] + MT_GEO_OFF);
            Geo* gd = (Geo*)((char*)R.tab + MT_GEO_OFF);
            T->nsys = n;
            T->pad = 0;
            memset((char*)R.htab[R.cur] + MT_CTR_OFF, 0, MT_GEO_OFF - MT_CTR_OFF);
            int64_t goff = 0;
            int cnt[MS_N];
            for (int st = 0; st < MS_N; st++) T->base[st][0] = 0;
            for (int i = 0; i < n; i++) {
                MJob& m = *act[a0 + i];
                cm_job* J = m.J;
                const cm_frames& fr = *m.fr;
                const int f0 = m.batches[r].first, F = m.batches[r].second;
                const double w = fr.weights[f0];
                if (J->pending && J->pending_w != w)
                    if (int e = flush(J, J->pending_w, R.stream)) return e;
                J->pending = true;
                J->pending_w = w;
                for (int f = 0; f < F; f++) {
                    cm::Cell64 c;
                    cm::cell_setup(fr.cells + 9 * (f0 + f), J->d.triclinic, &c);
                    J->volume_total += w * cm::cell_volume(c.H);
                }
                if (int e = batch_geo(J, F, fr.frame_index + f0, fr.cells + 9 * f0, m.cap, m.kcap, gh + goff)) return e;
                SysDev& S = T->sys[i];
                memset(&S, 0, sizeof(SysDev));
                S.P = J->kp;
                S.P.F = F;
                S.P.cap = (int)m.cap;
                S.P.kcap = (int)m.kcap;
                S.P.kcapr = (int)(m.kcap << (3 * S.P.ksub));
                S.P.mpt_auto = chunks_vary(S.P) ? 1 : 0;
                S.B = batch_bufs(J, gd + goff);
                S.B.dfield = (unsigned*)((char*)J->near.p + near_flags_bytes(F, m.cap));
                S.xu = (const char*)fr.d_x_solute + (size_t)f0 * J->Nu * 3 * ds;
                S.xv = (const char*)fr.d_x_solvent + (size_t)f0 * J->Nv * 3 * ds;
                S.zp[0] = (uint4*)J->cells_cnt.p;
                S.zp[1] = (uint4*)J->near.p;
                S.zp[2] = (uint4*)J->mcnt.p;
                S.z16[0] = (int64_t)(round16(sizeof(int) * (size_t)F * (m.cap + 1)) / 16);
                S.z16[1] = (int64_t)(near_bytes(F, m.cap) / 16);
                S.z16[2] = (int64_t)(round16(key_bytes(S.P, F)) / 16);
                stage_blocks(S.P, F, S.z16, S.nbx, cnt);
                for (int st = 0; st < MS_N; st++) T->base[st][i + 1] = T->base[st][i] + cnt[st];
                goff += F;
                J->frames += F;
            }
            HIPCHK(hipMemcpyAsync(R.tab, R.htab[R.cur], MT_GEO_OFF + sizeof(Geo) * (size_t)goff, hipMemcpyHostToDevice,
                                  R.stream));
            HIPCHK(hipEventRecord(R.up[R.cur], R.stream));
            R.cur ^= 1;
            if (R.graphs) {
                auto it = R.exec.find(variant);
                if (it == R.exec.end()) {
                    // first round of this variant: launched directly (which also
                    // settles the occupancy queries), captured from the next one
                    multi_launch_any(dtype, J0, R.stream, (const MultiTab*)R.tab, R.cus);
                    HIPCHK(hipGetLastError());
                    R.exec.emplace(variant, nullptr);
                    R.rounds++;
                    R.launches += MS_N + 2;
                    continue;
                }
                if (!it->second) {
                    hipGraph_t g = nullptr;
                    hipGraphExec_t x = nullptr;
                    HIPCHK(hipStreamBeginCapture(R.stream, hipStreamCaptureModeThreadLocal));
                    multi_launch_any(dtype, J0, R.stream, (const MultiTab*)R.tab, R.cus);
                    HIPCHK(hipStreamEndCapture(R.stream, &g));
                    HIPCHK(hipGraphInstantiate(&x, g, nullptr, nullptr, 0));
                    HIPCHK(hipGraphDestroy(g));
                    it->second = x;
                }
                HIPCHK(hipGraphLaunch(it->second, R.stream));
            } else {
                multi_launch_any(dtype, J0, R.stream, (const MultiTab*)R.tab, R.cus);
                HIPCHK(hipGetLastError());
            }
            R.rounds++;
            R.launches += MS_N + 2;
        }
    }
    return CM_OK;
}

}  // namespace

extern "C" {

int cm_jobs_submit_device(int32_t njobs, cm_job* const* jobs, const cm_frames* frames)
{
    if (njobs < 0 || (njobs > 0 && (!jobs || !frames))) return fail(CM_EINVAL, "null argument");
    for (int k = 0; k < njobs; k++) {
        cm_job* J = jobs[k];
        const cm_frames& fr = frames[k];
        if (!J) return fail(CM_EINVAL, "null job");
        if (J->finished) return fail(CM_ESTATE, "job already finished");
        for (int q = 0; q < k; q++)
            if (jobs[q] == J) return fail(CM_EINVAL, "a job appears twice");
        if (fr.nframes < 0 || (fr.nframes > 0 && (!fr.frame_index || !fr.d_x_solute || !fr.d_x_solvent || !fr.cells ||
                                                  !fr.weights)))
            return fail(CM_EINVAL, "invalid frame arrays");
        if (fr.dtype != CM_F64 && fr.dtype != CM_F32) return fail(CM_EINVAL, "dtype must be CM_F64 or CM_F32");
        for (int f = 0; f < fr.nframes; f++) {
            if (!(fr.weights[f] > 0.0) || !std::isfinite(fr.weights[f])) return fail(CM_EINVAL, "frame weights must be positive and finite");
            if (fr.frame_index[f] < 1 || fr.frame_index[f] > 0xFFFFFFFFll) return fail(CM_EINVAL, "frame_index must be in [1, 2^32)");
        }
    }
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= MR_MAX_DEVICES) return fail(CM_EUNSUPPORTED, "device index beyond the supported range");
    MultiRunner& R = multi_runners()[dev];
    std::lock_guard<std::mutex> lk(R.m);
    if (int r = multi_init(R)) return r;
    // the previous submission's rounds may still use buffers that are about
    // to grow
    HIPCHK(hipStreamSynchronize(R.stream));
    // groups of jobs sharing the kernel variant; the others run on their own.
    // The jobs of a submission hold their batch buffers at once: each gets an
    // equal share of MULTI_BUDGET for its frames per round (at least one).
    int nmulti = 0;
    for (int k = 0; k < njobs; k++)
        if (frames[k].nframes > 0 && jobs[k]->atoms_family && !jobs[k]->verify && !jobs[k]->arena && !jobs[k]->profiling)
            nmulti++;
    const int64_t share = MULTI_BUDGET / std::max(1, nmulti);
    std::map<int, std::vector<MJob>> groups;
    std::map<int, int> group_dtype;
    for (int k = 0; k < njobs; k++) {
        cm_job* J = jobs[k];
        const cm_frames& fr = frames[k];
        if (fr.nframes == 0) continue;
        if (!J->atoms_family || J->verify || J->arena || J->profiling) {
            if (int r = submit_common(J, fr.nframes, fr.frame_index, fr.d_x_solute, fr.d_x_solvent, fr.dtype, fr.cells,
                                      fr.weights, false))
                return r;
            continue;
        }
        const int ds = fr.dtype == CM_F32 ? 4 : 8;
        MJob m;
        m.J = J;
        m.fr = &fr;
        int64_t Fmax, pfb;
        if (int r = batch_plan(J, fr.nframes, fr.cells, ds, false, &m.cap, &m.kcap, &Fmax, &pfb)) return r;
        Fmax = std::max<int64_t>(1, std::min<int64_t>({Fmax, (int64_t)MS_FMAX, share / std::max<int64_t>(pfb, 1)}));
        // batches as the single-job path cuts them: equal batches over each
        // run of one frame weight
        int Fbig = 1;
        for (int f0 = 0; f0 < fr.nframes;) {
            const double w = fr.weights[f0];
            int run = 1;
            while (f0 + run < fr.nframes && fr.weights[f0 + run] == w) run++;
            const int nb = (int)((run + Fmax - 1) / Fmax);
            const int F = (run + nb - 1) / nb;
            for (int b = 0; b < run; b += F) m.batches.emplace_back(f0 + b, std::min(F, run - b));
            Fbig = std::max(Fbig, F);
            f0 += run;
        }
        // the job's own stream may still run earlier work on these buffers
        HIPCHK(hipStreamSynchronize(J->stream));
        if (int r = alloc_batch(J, Fbig, m.cap, m.kcap, ds, false)) return r;
        const int key = multi_variant(fr.dtype, J);
        groups[key].push_back(m);
        group_dtype[key] = fr.dtype;
    }
    for (auto& kv : groups)
        if (int r = multi_run_group(R, kv.second, group_dtype[kv.first])) return r;
    // the jobs' own streams (cm_job_finish, later submits) wait for the rounds
    HIPCHK(hipEventRecord(R.done, R.stream));
    for (auto& kv : groups)
        for (auto& m : kv.second) HIPCHK(hipStreamWaitEvent(m.J->stream, R.done, 0));
    return CM_OK;
}

int cm_multi_set_graphs(int32_t on)
{
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= MR_MAX_DEVICES) return fail(CM_EUNSUPPORTED, "device index beyond the supported range");
    MultiRunner& R = multi_runners()[dev];
    std::lock_guard<std::mutex> lk(R.m);
    R.graphs = on != 0;
    return CM_OK;
}

int cm_multi_stats(int64_t* rounds, int64_t* launches)
{
    if (!rounds || !launches) return fail(CM_EINVAL, "null argument");
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= MR_MAX_DEVICES) return fail(CM_EUNSUPPORTED, "device index beyond the supported range");
    MultiRunner& R = multi_runners()[dev];
    std::lock_guard<std::mutex> lk(R.m);
    *rounds = R.rounds;
    *launches = R.launches;
    return CM_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// entry point that allocates nothing (cm_mddf_noalloc)
// ---------------------------------------------------------------------------
// Fixed device scratch: every device buffer of such a call (integer hit
// counters, group maps, the batch buffers of the cell lists, placements and
// sorted molecules) is carved from it; the caller brings the coordinates and
// the FP64 output.  One copy per device, held until the process ends.
constexpr size_t SCRATCH_BYTES = (size_t)512 << 20;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

namespace {

constexpr int NA_MAX_DEVICES = 64;
// room for the 256-byte alignment of the carved buffers and the few bytes
// per frame (chunk offsets, drawn molecules) the per-frame estimate leaves out
constexpr int64_t NA_SLACK = 65536;

struct NoAllocDevice {
    std::mutex m;          // serialises the calls on this device
    bool ready = false;
    void* ptr = nullptr;   // device address of `scratch` on this device
    cm_job* job = nullptr; // host-side state reused by every call
};

NoAllocDevice* na_devices()
{
    static NoAllocDevice* d = new NoAllocDevice[NA_MAX_DEVICES];
    return d;
}

// device bytes a call needs: the integer counters and fixed buffers, plus
// the batch buffers of one frame
int64_t noalloc_fixed_bytes(const cm_job* J)
{
    int64_t b = 8 * J->acc_len + 8 * 4 * (int64_t)J->d.nbins + 64 + 4 * 256;
    if (J->d.groups_u_ptr) b += 4 * ((int64_t)J->d.natoms_per_mol_u + 2 + J->d.groups_u_ptr[J->d.natoms_per_mol_u]);
    if (J->d.groups_v_ptr) b += 4 * (J->Nv + 2 + J->d.groups_v_ptr[J->Nv]);
    return b;
}

}  // namespace

extern "C" {

int cm_mddf_noalloc(const cm_job_desc* desc, int32_t nframes, const int64_t* frame_index, const void* d_x_solute,
                    const void* d_x_solvent, int32_t dtype, const double* cells, const double* weights, double* d_acc,
                    double* volume_total, void* stream)
{
    if (!desc || !d_acc || !volume_total) return fail(CM_EINVAL, "null argument");
    if (nframes < 1 || !frame_index || !d_x_solute || !d_x_solvent || !cells || !weights)
        return fail(CM_EINVAL, "invalid frame arrays");
    if (dtype != CM_F64 && dtype != CM_F32) return fail(CM_EINVAL, "dtype must be CM_F64 or CM_F32");
    if (int r = validate_desc(*desc)) return r;
    for (int f = 0; f < nframes; f++) {
        if (!(weights[f] > 0.0) || !std::isfinite(weights[f])) return fail(CM_EINVAL, "frame weights must be positive and finite");
        if (frame_index[f] < 1 || frame_index[f] > 0xFFFFFFFFll) return fail(CM_EINVAL, "frame_index must be in [1, 2^32)");
    }
    // sizes first, on the host: a job that does not fit is refused before
    // any device work
    const int ds = dtype == CM_F32 ? 4 : 8;
    int64_t need_fixed, capmax, kcapmax, Fmax, pfb;
    {
        cm_job plan;
        plan.arena = (char*)1;   // (sized as the call below runs: from the scratch)
        job_params(&plan, *desc);
        need_fixed = noalloc_fixed_bytes(&plan);
        plan.d.memory_budget = (int64_t)SCRATCH_BYTES;
        if (int r = batch_plan(&plan, nframes, cells, ds, false, &capmax, &kcapmax, &Fmax, &pfb)) return r;
        if (need_fixed + pfb + NA_SLACK > (int64_t)SCRATCH_BYTES)
            return fail(CM_ENOMEM, "job too large for the no-allocation entry point: it needs " +
                                       std::to_string(need_fixed + pfb) + " bytes of device scratch for one frame, the "
                                       "fixed scratch holds " + std::to_string(SCRATCH_BYTES));
        Fmax = std::min<int64_t>(Fmax, std::max<int64_t>(1, ((int64_t)SCRATCH_BYTES - need_fixed - NA_SLACK) / pfb));
    }
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= NA_MAX_DEVICES) return fail(CM_EUNSUPPORTED, "device index beyond the supported range");
    NoAllocDevice& D = na_devices()[dev];
    std::lock_guard<std::mutex> lk(D.m);
    if (!D.ready) {
        // once per device, with that device current: the device address of
        // this device's copy of the scratch array
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return fail(CM_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        D.ptr = p;
        D.job = new cm_job();
        D.ready = true;
    }
    cm_job* J = D.job;
    // every buffer of the previous call is given up: the arena starts over
    DevBuf* bufs[] = {&J->cnt, &J->acc, &J->hits, &J->stats, &J->gmap, &J->geo, &J->cells_cnt, &J->cells_start,
                      &J->tmp4, &J->tmpcell, &J->sorted, &J->solw, &J->ucen, &J->vw, &J->vcell, &J->vcen, &J->P,
                      &J->vw_r, &J->vcen_r, &J->bflag, &J->blist, &J->nbulk, &J->uk, &J->drawn_ptr,
                      &J->drawn_idx, &J->xin_u, &J->xin_v, &J->near, &J->mkey, &J->mrank, &J->mcnt, &J->mstart, &J->msum,
                      &J->clmem, &J->msorted, &J->nnear, &J->chunk_base};
    for (DevBuf* b : bufs) *b = DevBuf{};
    J->arena = (char*)D.ptr;
    J->arena_cap = SCRATCH_BYTES;
    J->arena_used = 0;
    J->stream = (hipStream_t)stream;
    // the caller's output is the FP64 accumulator block (zeroed by the setup)
    const int64_t acc_len = 4 * (int64_t)desc->nbins + 2 * (int64_t)desc->n_groups_u * desc->nbins +
                            2 * (int64_t)desc->n_groups_v * desc->nbins;
    J->acc = DevBuf{d_acc, 8 * (size_t)acc_len};
    if (int r = job_setup(J, *desc)) return r;
    J->d.max_batch_frames = Fmax;
    J->d.memory_budget = (int64_t)SCRATCH_BYTES;
    // the batch buffers for the largest batch, carved once
    if (int r = alloc_batch(J, (int)Fmax, capmax, kcapmax, ds, false)) return r;
    if (int r = submit_common(J, nframes, frame_index, d_x_solute, d_x_solvent, dtype, cells, weights, false)) return r;
    if (J->pending) {
        if (int r = flush(J, J->pending_w)) return r;
        J->pending = false;
    }
    uint64_t gerr = 0;
    HIPCHK(hipMemcpyAsync(&gerr, (char*)J->stats.p + 16, 8, hipMemcpyDeviceToHost, J->stream));
    HIPCHK(hipStreamSynchronize(J->stream));
    J->finished = true;
    if (int r = geometry_error(gerr)) return r;
    *volume_total = J->volume_total;
    return CM_OK;
}

int cm_device_download(void* host, const void* dptr, size_t bytes)
{
    HIPCHK(hipMemcpy(host, dptr, bytes, hipMemcpyDeviceToHost));
    return CM_OK;
}

}  // extern "C"
