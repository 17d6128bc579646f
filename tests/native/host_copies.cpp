// Copies between node arrays and host memory on the HIP double: one check per run, named
// by the first argument.  Exit status 0: it holds.
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <future>
#include <map>
#include <memory>
#include <random>
#include <thread>

#include "../../droplet_amd/csrc/lattice_impl.h"

int copy_phi_plane(drp_lattice* L, int third, double* host, int* n1, int* n2);
void diag_free(drp_lattice*) {}  // the spectra's work space: not part of this program

using hip_double::rt;

namespace {

std::atomic<int> failures{0};
void check(bool ok, const char* what, const std::string& where) {
    if (!ok) {
        std::printf("%s: %s\n", where.c_str(), what);
        failures++;
    }
}

void done(int rc, const std::string& where) { check(rc == DRP_OK, drp_last_error(), where); }

drp_config config(int nx, int ny, int nz, int precision, int force = DRP_FORCE_NONE) {
    drp_config c;
    drp_config_default(&c);
    c.nx = nx;
    c.ny = ny;
    c.nz = nz;
    c.precision = precision;
    c.force_kind = force;
    return c;
}

std::vector<double> values(size_t n, unsigned seed, double lo, double hi) {
    std::mt19937 gen(seed);
    std::uniform_real_distribution<double> d(lo, hi);
    std::vector<double> v(n);
    for (double& x : v) x = d(gen);
    return v;
}

std::string where(const drp_lattice* L) {
    return std::to_string(L->cfg.nx) + "x" + std::to_string(L->cfg.ny) + "x" + std::to_string(L->cfg.nz) +
           (L->cfg.precision == DRP_FP64 ? " FP64" : " FP32");
}

// the lattice with random fields and populations, and a copy of every node value as the
// entry points must give it
struct State {
    drp_lattice* L = nullptr;
    std::vector<double> macro[5], pop[2], force[3];
    explicit State(const drp_config& c, unsigned seed = 1) {
        if (drp_create(&c, &L) != DRP_OK) {
            std::printf("create failed: %s\n", drp_last_error());
            std::exit(2);
        }
        const size_t n = (size_t)L->n;
        L->initialized = true;
        const bool f64 = c.precision == DRP_FP64;
        // a value of the arrays: a random number, for FP32 as the deviation from its reference
        auto fill = [&](void* base, int count, const double* ref, std::vector<double>* all, int first, unsigned s) {
            for (int a = 0; a < count; a++) {
                std::vector<double> v = values(n, s + a, 0.1, 1.0);
                for (size_t i = 0; i < n; i++) {
                    const size_t row = i / c.nx, at = (first + a) * L->G.ns + row * L->G.px + i % c.nx;
                    if (f64) {
                        ((double*)base)[at] = v[i];
                    } else {
                        ((float*)base)[at] = (float)v[i];
                        v[i] = ref[a] != 0.0 ? ref[a] + (double)(float)v[i] : (double)(float)v[i];
                    }
                }
                all->insert(all->end(), v.begin(), v.end());
            }
        };
        const double mref[5] = {c.phi1, 1.0 / 3.0, 0.0, 0.0, 0.0};
        for (int k = 0; k < 5; k++) fill(L->mac[L->cur], 1, &mref[k], &macro[k], k, seed * 100 + k);
        const double E[3] = {2.0 / 9.0, 1.0 / 9.0, 1.0 / 72.0}, F[3] = {-7.0 / 3.0, 1.0 / 3.0, 1.0 / 24.0};
        const double p0 = c.phi1 * c.T / (1.0 - c.b * c.phi1) - c.a * c.phi1 * c.phi1;
        double ref[2][15];
        for (int q = 0; q < 15; q++) {
            const int w = q == 0 ? 0 : (q <= 6 ? 1 : 2);
            ref[0][q] = (q == 0 ? c.phi1 : 0.0) + F[w] * p0;
            ref[1][q] = E[w];
        }
        for (int s = 0; s < 2; s++) fill(L->pop[L->cur], 15, ref[s], &pop[s], 15 * s, seed * 100 + 10 + 20 * s);
        if (L->force)
            for (int k = 0; k < 3; k++) force[k] = values(n, seed * 100 + 60 + k, -1.0, 1.0);
    }
    State(const State&) = delete;
    ~State() { drp_destroy(L); }

    // every output call gives the values (FP32 populations: the references' own rounding)
    void read(const char* what) const {
        const size_t n = (size_t)L->n;
        std::vector<double> out(15 * n);
        for (int k = 0; k < 5; k++) {
            done(drp_get_macro(L, k, out.data(), n), where(L));
            check(std::memcmp(out.data(), macro[k].data(), n * sizeof(double)) == 0, what, where(L) + " field");
        }
        for (int s = 0; s < 2; s++) {
            done(drp_get_populations(L, s, out.data(), 15 * n), where(L));
            double err = 0.0;
            for (size_t i = 0; i < 15 * n; i++) err = std::fmax(err, std::fabs(out[i] - pop[s][i]));
            check(err <= (L->cfg.precision == DRP_FP64 ? 0.0 : 1e-15), what, where(L) + " populations");
        }
        if (L->force) {
            done(drp_set_force(L, force[0].data(), force[1].data(), force[2].data(), n), where(L));
            std::vector<double> f[3];
            for (auto& v : f) v.resize(n);
            done(drp_get_force(L, f[0].data(), f[1].data(), f[2].data(), n), where(L));
            for (int k = 0; k < 3; k++) check(f[k] == force[k], what, where(L) + " force");
        }
    }

    // new fields and populations from the host
    void write(unsigned seed) {
        const size_t n = (size_t)L->n;
        for (int k = 0; k < 5; k++) macro[k] = values(n, seed + k, 0.1, 1.0);
        done(drp_init_fields(L, macro[0].data(), macro[1].data(), macro[2].data(), macro[3].data(), macro[4].data()), where(L));
        std::vector<double> out(n);
        for (int k = 0; k < 5; k++) {
            done(drp_get_macro(L, k, out.data(), n), where(L));
            check(out == macro[k], "fields set differ", where(L));
        }
        plane();
        for (int s = 0; s < 2; s++) {
            pop[s] = values(15 * n, seed + 10 + s, 0.1, 1.0);
            done(drp_set_populations(L, s, pop[s].data(), 15 * n), where(L));
        }
        for (int s = 0; s < 2; s++) {
            out.resize(15 * n);
            done(drp_get_populations(L, s, out.data(), 15 * n), where(L));
            check(out == pop[s], "populations set differ", where(L));
        }
    }

    // the deformation's plane (x, z) at y = 2
    void plane() const {
        const size_t nx = L->cfg.nx, ny = L->cfg.ny, nz = L->cfg.nz;
        std::vector<double> out(nx * nz);
        int n1 = 0, n2 = 0;
        done(copy_phi_plane(L, 2, out.data(), &n1, &n2), where(L));
        bool same = (size_t)n1 == nx && (size_t)n2 == nz;
        for (size_t z = 0; z < nz && same; z++)
            same = std::memcmp(&out[z * nx], &macro[0][nx * (2 + ny * z)], nx * sizeof(double)) == 0;
        check(same, "plane differs", where(L));
    }
};

// rows without and with padding; less and more than one thread's worth of populations
const int GRIDS[][3] = {{16, 7, 5}, {45, 22, 26}, {131, 70, 33}, {64, 96, 50}};

// A lattice of device 1 while the caller's current device is 0: everything that touches
// a stream or allocates has to run on the lattice's device, and the caller's stays.
void devices() {
    for (const auto& g : GRIDS)
        for (int precision : {DRP_FP64, DRP_FP32_SHIFTED}) {
            hipSetDevice(1);
            State s(config(g[0], g[1], g[2], precision, DRP_FORCE_FIELD));
            hipSetDevice(0);
            s.read("values differ");
            s.plane();
            check(hip_double::current == 0, "the caller's current device changed", where(s.L));
            for (auto& m : rt.live) check(m.second.host || m.second.dev == 1, "memory on another device", where(s.L));
        }
}

// What a kernel wrote to pinned memory is read after a wait that makes it visible.
void visibility() {
    for (const auto& g : GRIDS)
        for (int precision : {DRP_FP64, DRP_FP32_SHIFTED}) {
            State s(config(g[0], g[1], g[2], precision));
            s.read("values differ");
        }
}

// No pinned memory at all: the values come by the runtime's own copies.
void no_pinned_memory() {
    rt.pinned_limit = 0;
    for (const auto& g : GRIDS)
        for (int precision : {DRP_FP64, DRP_FP32_SHIFTED}) {
            State s(config(g[0], g[1], g[2], precision, DRP_FORCE_FIELD));
            s.read("values differ");
            if (precision == DRP_FP64) s.write(13);
            // FP64 values need no memory of the device on their way either
            if (precision == DRP_FP64) {
                State t(config(g[0], g[1], g[2], precision, DRP_FORCE_NONE));
                rt.device_limit = rt.device_bytes;
                t.read("values differ without device memory");
                t.write(14);
                rt.device_limit = SIZE_MAX;
            }
        }
}

// No device memory beyond the lattice's own: an FP64 lattice takes and gives everything.
void no_device_memory() {
    for (const auto& g : GRIDS) {
        State s(config(g[0], g[1], g[2], DRP_FP64, DRP_FORCE_FIELD));
        rt.device_limit = rt.device_bytes;
        s.read("values differ");
        s.plane();
        s.write(7);
        rt.device_limit = SIZE_MAX;
        check(hipGetLastError() == hipSuccess, "an error was left behind", where(s.L));
        s.write(8);
    }
}

// An error that an earlier HIP call of the caller's thread left behind is not a copy's.
void earlier_error() {
    for (const auto& g : GRIDS) {
        State s(config(g[0], g[1], g[2], DRP_FP64, DRP_FORCE_FIELD));
        const size_t n = (size_t)s.L->n;
        std::vector<double> out(15 * n);
        auto leave = [] { hip_double::last = hipErrorOutOfMemory; };
        leave();
        done(drp_get_macro(s.L, 0, out.data(), n), where(s.L));
        leave();
        done(drp_get_populations(s.L, 0, out.data(), 15 * n), where(s.L));
        leave();
        done(drp_set_force(s.L, s.force[0].data(), s.force[1].data(), s.force[2].data(), n), where(s.L));
        leave();
        done(drp_get_force(s.L, out.data(), out.data() + n, out.data() + 2 * n, n), where(s.L));
        leave();
        s.plane();
    }
}

// Transfers whose streams do not end hold as many chunks as they can get; one of another
// lattice ends all the same.
void independence() {
    const drp_config c = config(104, 104, 104, DRP_FP32_SHIFTED);  // 17 million values: eight threads
    std::vector<std::unique_ptr<State>> busy;
    std::vector<std::thread> threads;
    for (int k = 0; k < 3; k++) {
        busy.emplace_back(new State(c, 2 + k));
        busy.back()->L->stream->stall(true);
    }
    for (auto& b : busy) {
        drp_lattice* L = b->L;
        threads.emplace_back([L] {
            std::vector<double> out(15 * (size_t)L->n);
            done(drp_get_populations(L, 0, out.data(), out.size()), where(L));
        });
    }
    std::this_thread::sleep_for(std::chrono::seconds(1));
    State s(config(45, 22, 26, DRP_FP64));
    std::promise<void> ended;
    std::thread reader([&] {
        s.read("values differ");
        ended.set_value();
    });
    check(ended.get_future().wait_for(std::chrono::seconds(10)) == std::future_status::ready,
          "a transfer waited for other lattices' transfers", "independence");
    check(rt.pinned_blocks() <= 16, "more pinned memory than the pool's", "independence");
    for (auto& b : busy) b->L->stream->stall(false);
    for (auto& t : threads) t.join();
    reader.join();
    for (auto& b : busy) b->read("values differ");
}

// A deformation plane takes a plane's worth of device memory, not a lattice's; what needs
// more afterwards gets it.
void plane_memory() {
    for (const auto& g : GRIDS) {
        State s(config(g[0], g[1], g[2], DRP_FP64, DRP_FORCE_FIELD));
        rt.largest = 0;
        s.plane();
        check(rt.largest <= (size_t)g[0] * g[2] * sizeof(double), "more device memory than the plane", where(s.L));
        s.read("values differ");
        s.write(9);
    }
}

// A lattice whose arrays back to back just fit the device is made, without row padding
// and distances between arrays, and works.
void tight_lattice() {
    for (const auto& g : GRIDS)
        for (int precision : {DRP_FP64, DRP_FP32_SHIFTED}) {
            const size_t n = (size_t)g[0] * g[1] * g[2], value = precision == DRP_FP64 ? sizeof(double) : sizeof(float);
            rt.device_limit = 70 * n * value + drp::RANGE_WORDS * sizeof(uint64_t);
            {
                State s(config(g[0], g[1], g[2], precision));
                s.read("values differ");
            }
            rt.device_limit -= 1;
            const drp_config c = config(g[0], g[1], g[2], precision);
            drp_lattice* L = nullptr;
            check(drp_create(&c, &L) == DRP_ERR_ALLOC && !L, "a lattice that cannot fit was made", "tight lattice");
            rt.device_limit = SIZE_MAX;
        }
}

// The parts of a phi-range slot that a step uses follow the tiles of the default shape,
// also on thin lattices, and stay with the lattice: a step reads what the last one folded.
void range_parts() {
    const struct {
        int nx, ny, nz, precision, parts;
    } cases[] = {{16, 16, 16, DRP_FP64, 1},  {32, 32, 14, DRP_FP64, 1},          {32, 32, 16, DRP_FP64, 8},
                 {3, 3, 900, DRP_FP64, 8},   {17, 17, 28, DRP_FP64, 8},          {128, 64, 64, DRP_FP64, 8},
                 {130, 64, 64, DRP_FP64, 1}, {24, 24, 24, DRP_FP32_SHIFTED, 1},  {32, 32, 32, DRP_FP32_SHIFTED, 8},
                 {3, 3, 900, DRP_FP32_SHIFTED, 8}, {128, 128, 64, DRP_FP32_SHIFTED, 8}, {130, 128, 64, DRP_FP32_SHIFTED, 1}};
    for (const auto& k : cases) {
        const drp_config c = config(k.nx, k.ny, k.nz, k.precision);
        drp_lattice* L = nullptr;
        done(drp_create(&c, &L), "range parts");
        if (!L) continue;
        for (int shape = -1; shape < drp_tile_shape_count(); shape++) {
            if (shape >= 0) drp_set_tile_shape(L, shape);
            const int mask = k.precision == DRP_FP64 ? make_step_args(L, 1).range_mask : make_step_args32(L, 1).range_mask;
            check(mask == k.parts - 1, "wrong parts", where(L) + " shape " + std::to_string(shape));
        }
        drp_destroy(L);
    }
}

// Default tiles of a lattice with a force field, on both sides of the rule's lines.
void forced_tiles() {
    const struct {
        int nx, ny, nz, precision, shape;
    } cases[] = {{32, 32, 32, DRP_FP64, drp::SHAPE_32x4x2},         {33, 33, 33, DRP_FP64, drp::SHAPE_16x4x4},
                 {64, 32, 32, DRP_FP64, drp::SHAPE_32x4x2},         {100, 20, 28, DRP_FP64, drp::SHAPE_16x4x4},
                 {60, 20, 64, DRP_FP64, drp::SHAPE_32x4x2},         {256, 64, 64, DRP_FP64, drp::SHAPE_32x4x2},
                 {32, 32, 32, DRP_FP32_SHIFTED, drp::SHAPE_16x4x4}, {32, 32, 33, DRP_FP32_SHIFTED, drp::SHAPE_32x4x4}};
    for (const auto& k : cases)
        for (int force : {DRP_FORCE_FIELD, DRP_FORCE_NONE}) {
            const drp_config c = config(k.nx, k.ny, k.nz, k.precision, force);
            drp_lattice* L = nullptr;
            done(drp_create(&c, &L), "forced tiles");
            if (!L) continue;
            check(L->shape == (force == DRP_FORCE_FIELD ? k.shape : default_shape(k.precision)), "wrong tiles", where(L));
            drp_destroy(L);
        }
}

// Host arrays of a call go in together: through chunks (one launch where they fit one), or,
// where the arrays are long and few, by the runtime's copies and one launch that unpacks
// padded rows.
void together() {
    const struct {
        int nx, ny, nz, force_copies, force_launches, pop_copies, pop_launches;
    } cases[] = {{16, 7, 5, 0, 1, 0, 1}, {45, 22, 26, 0, 1, 0, 3}, {100, 50, 30, 3, 1, 0, 5}, {44, 40, 40, 3, 1, 1, 1},
                 {48, 40, 40, 3, 0, 1, 0}};
    for (const auto& k : cases) {
        State s(config(k.nx, k.ny, k.nz, DRP_FP64, DRP_FORCE_FIELD));
        const size_t n = (size_t)s.L->n;
        auto asked = [&](int copies, int launches, const char* what) {
            check(rt.copies == copies && rt.launches == launches,
                  (std::to_string(rt.copies) + " copies, " + std::to_string(rt.launches) + " launches").c_str(),
                  where(s.L) + " " + what);
            rt.copies = rt.launches = 0;
        };
        rt.copies = rt.launches = 0;
        done(drp_set_force(s.L, s.force[0].data(), s.force[1].data(), s.force[2].data(), n), where(s.L));
        asked(k.force_copies, k.force_launches, "force");
        done(drp_set_populations(s.L, 0, s.pop[0].data(), 15 * n), where(s.L));
        asked(k.pop_copies, k.pop_launches + 1, "populations");  // (and their moments)
        s.write(15);
    }
    // less memory than the runtime's copies ask for: an array at a time, then row by row
    State t(config(44, 40, 40, DRP_FP64, DRP_FORCE_FIELD));
    for (size_t room : {(size_t)8, (size_t)1, (size_t)0}) {
        if (t.L->pack) (void)hipFree(t.L->pack);
        t.L->pack = nullptr;
        t.L->pack_cap = 0;
        rt.device_limit = rt.device_bytes + room * (size_t)t.L->n * sizeof(double);
        t.write(16 + (unsigned)room);
        rt.device_limit = SIZE_MAX;
    }
}

const struct {
    const char* name;
    void (*run)();
} CHECKS[] = {{"devices", devices}, {"visibility", visibility}, {"no pinned memory", no_pinned_memory},
              {"no device memory", no_device_memory}, {"earlier error", earlier_error},
              {"independence", independence}, {"plane memory", plane_memory},
              {"tight lattice", tight_lattice}, {"range parts", range_parts},
              {"forced tiles", forced_tiles}, {"together", together}};

}  // namespace

int main(int argc, char** argv) {
    for (const auto& c : CHECKS)
        if (argc == 2 && std::string(argv[1]) == c.name) {
            c.run();
            std::map<std::string, int> kinds;
            for (const auto& v : rt.violations) kinds[v]++;
            for (const auto& v : kinds) check(false, (v.first + ", times " + std::to_string(v.second)).c_str(), c.name);
            for (const auto& m : rt.live) check(false, m.second.host ? "pinned memory left" : "device memory left", c.name);
            return failures ? 1 : 0;
        }
    return 3;
}
