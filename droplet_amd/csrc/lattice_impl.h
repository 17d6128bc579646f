// lattice_impl.h — internal state of a drp_lattice handle (not part of the ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>

#include "../../include/droplet.h"
#include "kernels.h"

struct drp_lattice {
    drp_config cfg{};
    drp::Phys phys{};
    int dev = 0;
    hipStream_t stream = nullptr;
    bool owns_stream = false;   // false for members of a batch (shared stream)
    bool host_io = false;       // counted by host_io_retain
    int64_t n = 0;         // nodes
    drp::Grid G{};         // layout of the population, field, force and tau arrays (choose_layout)
    int64_t step = 0;      // reference loop counter of the last completed step
    bool initialized = false;
    bool eq_init = false;  // populations are the equilibria of fields set by drp_init_* (no step since)
    int shape = 0;         // tile shape of the step kernel
    int range_mask = 0;    // parts of a phi-range slot that its steps use
    int cur = 0;           // which ping-pong buffer holds the current state
    void* pop[2] = {nullptr, nullptr};  // FP64: [f (15 G.ns) | g (15 G.ns)] doubles; FP32: floats
    void* mac[2] = {nullptr, nullptr};  // phi, p, u1, u2, u3 (5 G.ns)
    uint64_t* range = nullptr;          // 3 rotating slots of the phi range (RANGE_WORDS)
    double* tau = nullptr;              // LES relaxation-time field
    double* qh[2] = {nullptr, nullptr}; // non-equilibrium LES: sqrt(Pi:Pi) per node, with the populations' parity
    double* force = nullptr;            // FORCE_FIELD / SPECTRAL: fx | fy | fz
    double* spec = nullptr;             // SPECTRAL: transform work space and twiddle tables
    drp::SpectralWork specw{};
    double* spec_adv = nullptr;         // scale-separated advection: transform work space
    drp::SpectralWork specw_adv{};
    double* uadv = nullptr;             // scale-separated advection: band-passed u1 | u2 | u3
    double* pack = nullptr;             // one array (or plane) without row padding, on its way to or from the host
    size_t pack_cap = 0;                // its doubles
    double* tg = nullptr;               // Taylor-Green sin/cos tables
    double* partial = nullptr;          // diagnostics sums (REDUCE_WORK_DOUBLES)
    double* mac64 = nullptr;            // FP32 mode: FP64 copy of the macroscopic fields
    int* census = nullptr;              // droplet census work space (4 n + 4 ints, census.hip)
    double* budget = nullptr;           // energy-budget work space (7 n doubles + partial sums, budget.hip)
    struct drp_diag* diag = nullptr;    // plan and work space of the spectra (spectral_diag.hip)
    void* fp32_state = nullptr;         // FP32 mode: shift constants etc.
};

// The lattice's device, current for as long as one of these lives: copies between node
// arrays and the host are called from any thread, whose current device may be another,
// and launch kernels, record events and allocate.  A launch reports through the thread's
// last error, so one that an earlier call left there is cleared first: it is not the copy's.
class OnDevice {
  public:
    explicit OnDevice(int dev) {
        (void)hipGetLastError();
        if (hipGetDevice(&prev_) == hipSuccess && prev_ != dev) other_ = hipSetDevice(dev) == hipSuccess;
    }
    ~OnDevice() {
        if (other_) (void)hipSetDevice(prev_);
    }
    OnDevice(const OnDevice&) = delete;
    OnDevice& operator=(const OnDevice&) = delete;

  private:
    int prev_ = 0;
    bool other_ = false;
};

int drp_fail(int code, const char* fmt, ...);
drp::Phys make_phys(const drp_config& c);
int lattice_alloc(drp_lattice* L);
int lattice_create(const drp_config* cfg, hipStream_t stream, drp_lattice** out);
void lattice_free(drp_lattice* L);
drp::StepArgs make_step_args(drp_lattice* L, int64_t nstep);
int default_shape(int precision);
bool short_rows(const drp_config& c);  // 16x4x4 tiles suit the lattice better, by its rows
// SPECTRAL: recompute the force field from the current velocity (FP64 or FP32 fields)
int spectral_update(drp_lattice* L, int64_t nstep);
// scale-separated advection: the band-passed velocity the step's phi equilibria carry
int advect_update(drp_lattice* L, int64_t nstep);
int reset_range(drp_lattice* L);
// drp_stats from the compensated sums of the NPART diagnostics and the phi range slot
void stats_from_sums(const drp_lattice* L, const double* sums, const uint64_t* range_slot, drp_stats* st);
// LES tau for the next step: after a step (fresh = false, rank-block halos one
// step old) or for a replaced state (fresh = true, all neighbours current)
int les_update_tau(drp_lattice* L, bool fresh);

// host_io.hip: `count` node arrays (G.ns apart) to contiguous host arrays of n doubles;
// returns when they are there.  FP32 arrays hold deviations from ref.r[array].
struct HostRef {
    double r[15] = {};
};
int nodes_to_host(drp_lattice* L, const double* nodes, int count, double* host);
int nodes_to_host(drp_lattice* L, const float* nodes, int count, const HostRef& ref, double* host);
int dense_to_host(drp_lattice* L, const double* values, double* host);  // n values without gaps
// and `count` contiguous host arrays to node arrays, each where it lies or one behind the other
int nodes_from_host(drp_lattice* L, const double* const* host, int count, double* nodes);
int nodes_from_host(drp_lattice* L, const double* host, int count, double* nodes);
// a lattice that uses it exists, or no longer does
void host_io_retain();
void host_io_release();
// lattice.cpp: L->pack with room for that many doubles; null where there is no memory for it
double* pack_buffer(drp_lattice* L, size_t doubles);

// spectral_diag.hip
void diag_free(drp_lattice* L);

// deformation.cpp
int deformation(drp_lattice* L, int mode, double* Lo, double* Bo, double* Do);
// second-moment deformation (mode 2) of the current state and dD/dphi on its plane
// (n1 x n2 values, plane index third of the axis that is neither x nor wall-normal)
int deformation_inertia_grad(drp_lattice* L, double* D, double* grad, int* n1, int* n2, int* third);
int copy_phi_plane(drp_lattice* L, int third, double* host, int* n1, int* n2);

// fp32_shifted.cpp
int fp32_init_from_host_fields(drp_lattice* L, const double* const* host);
int fp32_step(drp_lattice* L, int nsteps);
drp::StepArgs32 make_step_args32(drp_lattice* L, int64_t nstep);
int fp32_get_macro(drp_lattice* L, int field, double* host);
int fp32_get_populations(drp_lattice* L, int set, double* host);
int fp32_set_populations(drp_lattice* L, int set, const double* host, int which);
int fp32_macro_fp64_view(drp_lattice* L, const double** mac);
