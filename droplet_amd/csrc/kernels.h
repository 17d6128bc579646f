// kernels.h — launch interfaces between the C-ABI host code and the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace drp {

enum { FORCE_NONE = 0, FORCE_TAYLOR_GREEN = 1, FORCE_FIELD = 2 };

// Map the linear workgroup id to a tile so that each XCD (workgroups are dealt
// round-robin to the 8 XCDs) gets a contiguous block of tiles: neighbouring
// tiles, which share halo lines, then share one L2.  Where the number of workgroups is no
// multiple of 8 the id is the tile, and neighbours lie on different XCDs (a launch may
// round its number up: adjoint.hip).
__device__ __forceinline__ int xcd_tile(int b, int nb) {
    if ((nb & 7) != 0) return b;
    return (b & 7) * (nb >> 3) + (b >> 3);
}
// How the node arrays of a lattice lie in memory: rows of nx elements px apart
// (px >= nx), arrays ns apart.  What lies between rows and arrays is never read as
// a node.
struct Grid {
    int nx, ny, nz;
    int px;      // elements from one x row to the next
    int64_t ns;  // elements from one array to the next
    // elements of one array, row padding included
    __host__ __device__ __forceinline__ int64_t slots() const { return (int64_t)px * ny * nz; }
    __host__ __device__ __forceinline__ int64_t node(int x, int y, int z) const {
        return x + (int64_t)px * (y + (int64_t)ny * z);
    }
    // node of coordinates up to one period outside the lattice (periodic wrap)
    __device__ __forceinline__ int64_t at(int x, int y, int z) const {
        x = x < 0 ? x + nx : (x >= nx ? x - nx : x);
        y = y < 0 ? y + ny : (y >= ny ? y - ny : y);
        z = z < 0 ? z + nz : (z >= nz ? z - nz : z);
        return node(x, y, z);
    }
};

// The global phi range of a step lives in one of three rotating slots, as
// order-preserving integers (d3q15.h).  A slot is kept in parts, 256 bytes apart,
// each folded into by every eighth workgroup with atomics: on one pair of addresses
// the workgroups of a small lattice, which end together, queue.  Step with one and with
// eight parts, us: FP64 98 tiles (28^3) 12.2 and 11.2, 128 (32^3) 12.8 and 10.8, 1024
// (64^3) 40.5 and 37.7; FP32 64 tiles (32^3) 11.0 and 10.2, 512 (64^3) 23.6 and 18.1,
// 1728 (96^3) 65.3 and 62.9.  With many more tiles than fit the card at once their
// workgroups end at different times, eight parts bring nothing, and a step that reads the
// range pays for eight loads in each workgroup: with the viscosity of phi FP64 2904 tiles
// (88^3) 101.1 and 102.4, FP32 2704 (104^3) 103.4 and 105.6; 256^3 1984 and 2023.  With
// few tiles it pays without a queue: FP32 36 tiles (24^3) 11.1 and 11.5, FP64 50 (20^3)
// 11.6 and 12.1.  On both sides only part 0 takes the folds of a step and only it is read
// by one.  The parts that take none hold the limits that a slot is reset to, or a range
// set on all parts, so that the fold over all of them is the range at every size.
constexpr int RANGE_PARTS = 8, RANGE_PART_WORDS = 32;
constexpr int RANGE_SLOT_WORDS = RANGE_PARTS * RANGE_PART_WORDS;
constexpr int RANGE_WORDS = 3 * RANGE_SLOT_WORDS;
constexpr int64_t RANGE_PARTS_MIN_TILES = 64, RANGE_PARTS_MAX_TILES = 2048;
// a lattice's mask of parts, RANGE_PARTS - 1 or 0, from the tiles of its default shape: a
// step reads the parts that the step before it folded into, so it does not follow a later
// change of the shape
inline int range_mask(int64_t tiles) {
    return tiles >= RANGE_PARTS_MIN_TILES && tiles <= RANGE_PARTS_MAX_TILES ? RANGE_PARTS - 1 : 0;
}
// (max, min) of a slot; a step passes its mask
__device__ __forceinline__ void range_words(const uint64_t* __restrict__ range, int slot, uint64_t& mx, uint64_t& mn,
                                            int mask = RANGE_PARTS - 1) {
    const uint64_t* r = range + slot * RANGE_SLOT_WORDS;
    if (mask == 0) {
        mx = r[0];
        mn = r[1];
        return;
    }
    // part 0 is read with the others: read before the branch, they would wait for it
    uint64_t a[RANGE_PARTS], b[RANGE_PARTS];
#pragma unroll
    for (int p = 0; p < RANGE_PARTS; p++) {
        a[p] = r[p * RANGE_PART_WORDS];
        b[p] = r[p * RANGE_PART_WORDS + 1];
    }
    mx = a[0];
    mn = b[0];
#pragma unroll
    for (int p = 1; p < RANGE_PARTS; p++) {
        mx = a[p] > mx ? a[p] : mx;
        mn = b[p] < mn ? b[p] : mn;
    }
}
// set part p of a slot
__device__ __forceinline__ void range_set_part(uint64_t* range, int slot, int p, uint64_t mx, uint64_t mn) {
    range[slot * RANGE_SLOT_WORDS + p * RANGE_PART_WORDS] = mx;
    range[slot * RANGE_SLOT_WORDS + p * RANGE_PART_WORDS + 1] = mn;
}
// fold a workgroup's (max, min) into its part of a slot
__device__ __forceinline__ void range_fold(uint64_t* range, int slot, int mask, uint64_t mx, uint64_t mn) {
    uint64_t* r = range + slot * RANGE_SLOT_WORDS + (blockIdx.x & mask) * RANGE_PART_WORDS;
    atomicMax(reinterpret_cast<unsigned long long*>(r), (unsigned long long)mx);
    atomicMin(reinterpret_cast<unsigned long long*>(r + 1), (unsigned long long)mn);
}

// batched launch: per-instance step arguments and first-tile offsets in device memory
struct BatchLaunch {
    const void* args;      // StepArgs[ninst] or StepArgs32[ninst]
    const int* tile_start; // [ninst], ascending, tile_start[0] = 0
    int ninst;
    int total_tiles;
};

// tile shapes of the step kernel (nodes per workgroup in x, y, z; two threads per node)
enum { SHAPE_16x4x4 = 0, SHAPE_32x4x2 = 1, SHAPE_64x2x2 = 2, SHAPE_32x2x4 = 3, SHAPE_32x4x4 = 4, SHAPE_32x8x2 = 5,
       SHAPE_64x4x2 = 6, SHAPE_COUNT = 7 };
constexpr int SHAPE_DIMS[SHAPE_COUNT][3] = {{16, 4, 4}, {32, 4, 2}, {64, 2, 2}, {32, 2, 4},
                                            {32, 4, 4}, {32, 8, 2}, {64, 4, 2}};

// tile counts and wrap mode of one lattice for a tile shape
template <typename A> inline void set_tiles(A& a, int TX, int TY, int TZ) {
    a.tiles_x = (a.nx + TX - 1) / TX;
    a.tiles_y = (a.ny + TY - 1) / TY;
    a.tiles_z = (a.nz + TZ - 1) / TZ;
    a.wrap_mod = (a.nx <= TX || a.ny <= TY || a.nz <= TZ) ? 1 : 0;
}

// Physical constants of one lattice as the kernels need them.
struct Phys {
    double tau_f;     // phi-population relaxation time
    double kf, kf6;   // kappa_f and kappa_f/6 (the reference folds kappaf/6.0d0 at compile time)
    double kg;        // kappa_g
    double T, a, b;   // van der Waals constants
    double nu1, dnu;  // nu1 and nu2 - nu1
    double phi1, phi2;
    double tg_amp;    // Taylor-Green force amplitude
    double les_c;     // Cs*Cs*Delta*Delta (evaluated left to right)
    int les;          // Smagorinsky on
};

struct StepArgs {
    int nx, ny, nz;
    int tiles_x, tiles_y, tiles_z;
    int px;               // row pitch (Grid)
    int64_t ns;           // elements from one population, field or force array to the next
    const double* f_in;   // [15][ns] phi populations (reference f)
    const double* g_in;   // [15][ns] momentum populations (reference g)
    double* f_out;
    double* g_out;
    const double* mac_in; // phi, p, u1, u2, u3 (5 x ns)
    double* mac_out;
    const double* tau_field;              // LES: tau_g per node, else nullptr
    const double *fx, *fy, *fz;           // FORCE_FIELD
    const double *sinx, *cosx, *sinz, *cosz;  // FORCE_TAYLOR_GREEN tables
    double tau_f, kf, kf6, kg, T, a, b, nu1, dnu, tg_amp, phi1, phi2;
    double tau_const;     // tau_g when nu1 == nu2: 0.5 + 3 nu1
    double ekf[3], ekg[3];  // E kappa_f, E kappa_g for the rest, axis and diagonal weights
    double wall_u_now;
    int wall_axis;        // 0, 2 (y) or 3 (z)
    int force_kind;
    uint64_t* range;      // RANGE_WORDS
    int slot_read, slot_write, slot_reset;
    int range_mask;       // parts of a slot that a step uses
    int wrap_mod;         // set by the launcher: a grid extent does not exceed the tile extent
    int model;            // 0 free energy (phi populations), 1 Allen-Cahn (phi stencil update)
    double ac_a, ac_m, ac_w;  // Allen-Cahn A, mobility M = (1 - A)/6, interface width W
    // non-equilibrium Smagorinsky: sqrt(Pi:Pi) per node from the last step (in) and
    // of this step (out); 18 Cs^2 D^2, 6 Cs^2 D^2, Cs^2 D^2 (left to right)
    const double* qh_in;
    double* qh_out;
    double neq_c18, neq_c6, neq_cc;
    // scale-separated advection: the velocity the phi equilibria carry (u1 | u2 | u3),
    // or nullptr for u itself
    const double* uadv;
};

hipError_t launch_step_fp64(const StepArgs& a, int shape, hipStream_t st, const BatchLaunch* batch = nullptr);

// FP32 shifted storage (step_fp32.hip): populations and fields as FP32
// deviations from the continuous phase at rest
struct StepArgs32 {
    int nx, ny, nz;
    int tiles_x, tiles_y, tiles_z;
    int px;
    int64_t ns;
    const float* f_in;
    const float* g_in;
    float* f_out;
    float* g_out;
    const float* mac_in;   // phi - phi1, p - 1/3, u1, u2, u3
    float* mac_out;
    const float* tau_field;
    const double *fx, *fy, *fz;
    const double *sinx, *cosx, *sinz, *cosz;
    double tg_amp, phi1, phi2;
    float phi1f, Tf, af, bf, one_m_bphi1, kff, kf6f, kgf;
    float rtau_f, rtau_const, nu1f, dnuf;
    float wall_u_now;
    int wall_axis, force_kind;
    uint64_t* range;
    int slot_read, slot_write, slot_reset;
    int range_mask;       // parts of a slot that a step uses
    int wrap_mod;
};
hipError_t launch_step_fp32(const StepArgs32& a, int shape, hipStream_t st, const BatchLaunch* batch = nullptr);

// Rank blocks of the reference's LES decomposition, in nodes per axis (all 0:
// none).  grad u for the eddy viscosity takes every neighbour outside a node's
// block, periodic wraps included, from the state the step started from.
struct LesBlocks {
    int bx, by, bz;
};

// conversions between FP64 absolute and FP32 shifted representations; fref is
// the 15 reference phi populations H_q phi1 + F_q p0(phi1) (host-computed)
struct ShiftRef {
    double fr[15];
    double phi1;
};
hipError_t launch_to_shifted(const Grid& G, const ShiftRef& r, const double* pop64, const double* mac64, float* pop32,
                             float* mac32, hipStream_t st);
hipError_t launch_pops_to_shifted(const Grid& G, const ShiftRef& r, const double* pop64, float* pop32, int set,
                                  hipStream_t st);
hipError_t launch_macro_from_shifted(const Grid& G, double phi1, const float* mac32, double* mac64, hipStream_t st);
hipError_t launch_moments_fp32(const Grid& G, const float* f, const float* g, float* mac, int which, hipStream_t st);
// Planes a workgroup of the LES kernels marches over: 16 where that leaves four
// workgroups per CU, else fewer, down to 2.  A short march reads its two halo planes more
// often, from L2, but a small lattice leaves most CUs idle with a long one.  Spectral-forced
// step with 16 and with this: FP64 92 and 71 us at 64^3, 186 and 180 at 96^3, 351 and 346 at
// 128^3; FP32 67 and 52, 225 and 222 at 64^3 and 128^3; the same from 192^3 on.
constexpr int LES_ZC_MIN = 2, LES_BLOCKS = 1024;
inline int les_planes(int columns, int nz) {
    int zc = 16;
    while (zc > LES_ZC_MIN && (int64_t)columns * ((nz + zc - 1) / zc) < LES_BLOCKS) zc /= 2;
    return zc;
}
hipError_t launch_les_tau_fp32(const Grid& G, const Phys& ph, const float* mac, const float* mac_old,
                               const LesBlocks& blk, const uint64_t* range, int slot, float* tau, hipStream_t st);

// populations := equilibria of the macroscopic fields (ini, program/lbm_drop_xy.f90:244-251)
hipError_t launch_init_equilibrium_fp64(const Grid& G, const Phys& ph, const double* mac, double* f,
                                        double* g, hipStream_t st);
// recompute moments from populations: which & 1 -> phi from f, which & 2 -> p, u from g
hipError_t launch_moments_fp64(const Grid& G, const double* f, const double* g, double* mac, int which,
                               hipStream_t st);
// Smagorinsky tau field for the next step (program/LES_drop.f90:598-693) from the
// state a step left (mac), the one it started from (mac_old, read across rank
// blocks) and that step's phi range slot
hipError_t launch_les_tau_fp64(const Grid& G, const Phys& ph, const double* mac, const double* mac_old,
                               const LesBlocks& blk, const uint64_t* range, int slot, double* tau, hipStream_t st);
// derived fields of the analysis programs (budget.hip): kind = DRP_DERIVED_*; rows of
// the result `pitch` doubles apart
hipError_t launch_derived_fp64(const Grid& G, const Phys& ph, const double* mac, int kind, double* out, int64_t pitch, hipStream_t st);

// diagnostics sums: NPART doubles per workgroup (at most REDUCE_MAX_BLOCKS), then at
// work[REDUCE_OUT] the NPART total sums and the two words of the phi range slot
constexpr int NPART = 10;
constexpr int REDUCE_MAX_BLOCKS = 2048;
constexpr int REDUCE_OUT = REDUCE_MAX_BLOCKS * NPART;
constexpr int REDUCE_WORK_DOUBLES = REDUCE_OUT + 16;
hipError_t launch_reduce_fp64(const Grid& G, const Phys& ph, const double* mac, const uint64_t* range, int slot,
                              double* work, hipStream_t st);
// rows of nx doubles, `stride` apart, to contiguous rows
hipError_t launch_pack_rows(int nx, int64_t rows, int64_t stride, const double* nodes, double* packed, hipStream_t st);
// fill a range slot with (max, min) = (vmax, vmin)
hipError_t launch_range_set(uint64_t* range, int slot, double vmax, double vmin, hipStream_t st);

// spectral.hip: linear forcing of the shells 1 <= |k| < kc from the velocity field
struct SpectralWork {
    double2 *A, *B, *C;       // forward transform stages
    double2 *twx, *twy, *twz; // e^{2 pi i j / n} tables
    double* elow;             // energy of the forced shells (last call)
};
size_t spectral_work_doubles(int nx, int ny, int nz, int kc);
void spectral_work_layout(SpectralWork& w, double* base, int nx, int ny, int nz, int kc);
hipError_t launch_spectral_force(const SpectralWork& w, const Grid& G, int kc, double eps, const double* u1,
                                 const double* u2, const double* u3, double* fx, double* fy, double* fz,
                                 hipStream_t st);
hipError_t launch_spectral_force(const SpectralWork& w, const Grid& G, int kc, double eps, const float* u1,
                                 const float* u2, const float* u3, double* fx, double* fy, double* fz,
                                 hipStream_t st);
// band-pass of u keeping the shells klo <= int|k| < khi (2 <= khi <= 5; work space of kc = khi)
hipError_t launch_spectral_band(const SpectralWork& w, const Grid& G, int klo, int khi, const double* u1,
                                const double* u2, const double* u3, double* o1, double* o2, double* o3,
                                hipStream_t st);

// adjoint.hip: one reverse step of the FP64 step (equal viscosities, no LES)
struct AdjArgs {
    Grid G;
    const double* f;        // forward phi populations at step n (15 ns)
    const double* mac;      // forward macroscopic fields at step n (5 ns)
    const double* Fin;      // adjoint of f^{n+1} without its stencil part (15 ns)
    const double* phin_in;  // stencil part of the adjoint of phi^{n+1} (n)
    const double* Gin;      // adjoint of g^{n+1} (15 ns)
    double* Fout;           // adjoint of f^n without its stencil part
    double* Gout;           // adjoint of g^n
    double* lapA;           // adjoint of lap phi at step n (n)
    double* gradA;          // adjoint of grad phi at step n (3 ns)
    double* acc;            // [tiles][3]: d/dtau_f, d/dkappa_g, d/dU_wall, accumulated
    double tau_f, tau_g, kf, kf6, kg, T, a, b;
    double rtau_f, rtau_g, rtau_f2;  // 1 / tau_f, 1 / tau_g, 1 / (tau_f tau_f)
    double om_f, om_g;               // 1 - 1 / tau_f, 1 - 1 / tau_g
    int wall_axis;          // 0, 2 (y) or 3 (z)
    int wall_active;        // the walls move during step n -> n+1
    int first;              // step n is the initial equilibrium of constant fields
};
int adj_block_count(const Grid& G);
hipError_t launch_adj_collide_fp64(const AdjArgs& a, hipStream_t st);
hipError_t launch_adj_stencil_fp64(const Grid& G, const double* lapA, const double* gradA, double* out,
                                   hipStream_t st);
hipError_t launch_adj_seed_area_fp64(const Grid& G, const double* phi, double w, double* lapA,
                                     double* gradA, hipStream_t st);
hipError_t launch_adj_add_plane(const Grid& G, int n1, int n2, int wall_y, int third, const double* vals,
                                double* out, hipStream_t st);

}  // namespace drp
