// aux_kernels.hip — initialisation, moment recomputation, LES relaxation-time
// field and diagnostics reductions (FP64).  None of these is on the per-step hot
// path except the LES tau field, the eddy-viscosity part of the reference
// `physics` (program/LES_drop.f90:598-693), computed after each step.
#include <algorithm>

#include "d3q15.h"
#include "kernels.h"

namespace drp {

template <int Q0, int Q1, typename Fn> __device__ __forceinline__ void sfor(Fn&& fn) {
    if constexpr (Q0 < Q1) {
        fn(std::integral_constant<int, Q0>{});
        sfor<Q0 + 1, Q1>(fn);
    }
}

// lap phi and grad phi at (x,y,z) from global memory (various_cal :608-633)
__device__ void phi_stencil(const Grid& G, const double* phi, int x, int y, int z, double& lap, double& g0,
                            double& g1, double& g2) {
    lap = -14.0 * phi[G.at(x, y, z)];
    g0 = g1 = g2 = 0.0;
    sfor<1, 15>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        using D = Dir<q>;
        const double v = phi[G.at(x + D::cx, y + D::cy, z + D::cz)];
        lap = lap + v;
        g0 = acc<D::cx>(g0, v);
        g1 = acc<D::cy>(g1, v);
        g2 = acc<D::cz>(g2, v);
    });
    lap = lap / 5.0;
    g0 = g0 / 10.0;
    g1 = g1 / 10.0;
    g2 = g2 / 10.0;
}

// True when the neighbour (xx, yy, zz) (not wrapped) of node (x, y, z) lies
// outside the node's rank block: program/LES_drop.f90 (:153-157) and
// LES_drop_xy.f90 (:150-153) take every such neighbour from the halo exchanged
// at the start of the step.  B.bx = 0: no decomposition, every neighbour current.
__device__ __forceinline__ bool les_halo(const LesBlocks& B, int x, int y, int z, int xx, int yy, int zz) {
    if (B.bx == 0) return false;
    const int x0 = (x / B.bx) * B.bx, y0 = (y / B.by) * B.by, z0 = (z / B.bz) * B.bz;
    return xx < x0 || xx >= x0 + B.bx || yy < y0 || yy >= y0 + B.by || zz < z0 || zz >= z0 + B.bz;
}

__global__ void init_equilibrium_fp64(Grid G, Phys P, const double* __restrict__ mac, double* __restrict__ f,
                                      double* __restrict__ g) {
    const int64_t N = G.ns, s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int x = s % G.px, y = (s / G.px) % G.ny, z = s / ((int64_t)G.px * G.ny);
    if (x >= G.nx || z >= G.nz) return;
    NodeEq<double> nd;
    nd.phi = mac[s];
    nd.p = mac[N + s];
    nd.u1 = mac[2 * N + s];
    nd.u2 = mac[3 * N + s];
    nd.u3 = mac[4 * N + s];
    double lap;
    phi_stencil(G, mac, x, y, z, lap, nd.g0, nd.g1, nd.g2);
    const double ph = nd.phi;
    const double p0 = ph * P.T / (1.0 - P.b * ph) - P.a * (ph * ph);
    nd.A = p0 - P.kf * ph * lap - P.kf6 * (nd.g0 * nd.g0 + nd.g1 * nd.g1 + nd.g2 * nd.g2);
    const double usq = nd.u1 * nd.u1 + nd.u2 * nd.u2 + nd.u3 * nd.u3;
    const double s2h = 1.5 * (nd.g0 * nd.g0 + nd.g1 * nd.g1 + nd.g2 * nd.g2);
    sfor<0, 15>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        const double gt = korteweg<q>(nd.g0, nd.g1, nd.g2, s2h);
        f[q * N + s] = feq<q>(nd, gt, ekappa<q>(P.kf));
        g[q * N + s] = geq<q>(nd, usq, gt, ekappa<q>(P.kg));
    });
}

__global__ void moments_fp64(Grid G, const double* __restrict__ f, const double* __restrict__ g,
                             double* __restrict__ mac, int which) {
    const int64_t N = G.ns, s = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (s >= G.slots()) return;
    double ph = f[s], pr = g[s] / 3.0, m1 = 0.0, m2 = 0.0, m3 = 0.0;
    sfor<1, 15>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        using D = Dir<q>;
        const double gv = g[q * N + s];
        ph = ph + f[q * N + s];
        pr = pr + gv / 3.0;
        m1 = acc<D::cx>(m1, gv);
        m2 = acc<D::cy>(m2, gv);
        m3 = acc<D::cz>(m3, gv);
    });
    if (which & 1) mac[s] = ph;
    if (which & 2) {
        mac[N + s] = pr;
        mac[2 * N + s] = m1;
        mac[3 * N + s] = m2;
        mac[4 * N + s] = m3;
    }
}

// LES tau tiles of LES_TX x LES_TY x LES_TZ nodes, one node per thread
constexpr int LES_TX = 32, LES_TY = 4, LES_TZ = 2;
// periodic index of v in [-1, n + tile): one conditional add or subtract, or a
// full modulo where a tile is longer than the grid (small)
__device__ __forceinline__ int wrap_any(int v, int n, bool small) {
    if (small) return ((v % n) + n) % n;
    return v < 0 ? v + n : (v >= n ? v - n : v);
}

// tau_g for the next step from the state a step left (mac: phi, p, u of this
// step; mac_old: the state the step started from) and that step's phi range:
// grad u as grad_u_cal takes it at the end of physics (:447-477, :660), with
// the neighbours outside a node's rank block from mac_old (les_halo), then
// nu_e = Cs^2 Delta^2 sqrt(2 S:S) with S_ab = 0.5 (d_b u_a + d_a u_b) (strain_cal
// :479-499, :661-677; amdflang lowers **0.5d0 to sqrt) and tau = 0.5 + 3 (nu + nu_e)
// (:679-690).  mac_old == mac gives the tau of a state with current halos (ini_op).
// u (and, with rank blocks, the old u) of a tile and its 1-node halo are staged
// in LDS once per workgroup.
template <bool STALE>
__global__ __launch_bounds__(LES_TX* LES_TY* LES_TZ) void les_tau_fp64(Grid G, Phys P, const double* __restrict__ mac,
                                                                       const double* __restrict__ mac_old, LesBlocks B,
                                                                       const uint64_t* __restrict__ range, int slot,
                                                                       double* __restrict__ tau, int tiles_x,
                                                                       int tiles_y) {
    constexpr int HX = LES_TX + 2, HY = LES_TY + 2, HZ = LES_TZ + 2, H = HX * HY * HZ, NT = LES_TX * LES_TY * LES_TZ;
    __shared__ double su[3][H];
    __shared__ double so[STALE ? 3 : 1][STALE ? H : 1];
    const int64_t N = G.ns;
    const int tile = blockIdx.x;
    const int x0 = (tile % tiles_x) * LES_TX, y0 = ((tile / tiles_x) % tiles_y) * LES_TY,
              z0 = (tile / (tiles_x * tiles_y)) * LES_TZ;
    const bool small = G.nx <= LES_TX || G.ny <= LES_TY || G.nz <= LES_TZ;
    for (int h = threadIdx.x; h < H; h += NT) {
        const int hx = h % HX, hy = (h / HX) % HY, hz = h / (HX * HY);
        const int64_t g = G.node(wrap_any(x0 + hx - 1, G.nx, small), wrap_any(y0 + hy - 1, G.ny, small),
                                 wrap_any(z0 + hz - 1, G.nz, small));
        for (int k = 0; k < 3; k++) {
            su[k][h] = mac[(2 + k) * N + g];
            if constexpr (STALE) so[k][h] = mac_old[(2 + k) * N + g];
        }
    }
    __syncthreads();
    const int tx = threadIdx.x % LES_TX, ty = (threadIdx.x / LES_TX) % LES_TY, tz = threadIdx.x / (LES_TX * LES_TY);
    const int x = x0 + tx, y = y0 + ty, z = z0 + tz;
    if (x >= G.nx || y >= G.ny || z >= G.nz) return;
    const int64_t s = G.node(x, y, z);
    double gu[3][3];
    for (int k = 0; k < 3; k++)
        for (int a = 0; a < 3; a++) gu[k][a] = 0.0;
    sfor<1, 15>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        using D = Dir<q>;
        const int h = (tx + 1 + D::cx) + HX * ((ty + 1 + D::cy) + HY * (tz + 1 + D::cz));
        const bool old = STALE && les_halo(B, x, y, z, x + D::cx, y + D::cy, z + D::cz);
        for (int k = 0; k < 3; k++) {
            const double v = old ? so[STALE ? k : 0][STALE ? h : 0] : su[k][h];
            gu[k][0] = acc<D::cx>(gu[k][0], v);
            gu[k][1] = acc<D::cy>(gu[k][1], v);
            gu[k][2] = acc<D::cz>(gu[k][2], v);
        }
    });
    for (int k = 0; k < 3; k++)
        for (int a = 0; a < 3; a++) gu[k][a] = gu[k][a] / 10.0;
    // S_ab = 0.5 (d_b u_a + d_a u_b), nu_e = Cs^2 Delta^2 sqrt(2 S:S)  (:671-675, strain :481-501)
    double sum = 0.0;
    for (int b = 0; b < 3; b++)
        for (int a = 0; a < 3; a++) {
            const double sab = 0.5 * (gu[a][b] + gu[b][a]);
            sum = sum + sab * sab;
        }
    const double nue = P.les_c * sqrt(2.0 * sum);
    uint64_t mx_bits, mn_bits;
    range_words(range, slot, mx_bits, mn_bits);
    const double rmax = from_ordered_bits(mx_bits), rmin = from_ordered_bits(mn_bits);
    const double rg = rmax - rmin;
    double frac = (mac[s] - rmin) / rg;
    if (rg == 0.0) frac = 0.0;
    const double nu = frac * P.dnu + P.nu1;
    tau[s] = 0.5 + 3.0 * (nu + nue);
}

// The same tau with every neighbour current (no rank blocks), marching in z: a
// workgroup owns a ZM_TX x ZM_TY column of nodes over zc planes and keeps the
// planes z-1, z, z+1 of u (with a one-node x-y halo) in a ring of three LDS
// planes.  While plane z is computed, the loads of plane z+2 are already in
// flight into registers (stored into the ring slot of plane z-1 afterwards), so
// their latency overlaps the stencil work.  u is read from L2 / HBM about
// (66 x 10)/(64 x 8) (zc + 2)/zc times.  Sums are formed in the order of
// les_tau_fp64 (the divisions by 10 correctly rounded), so both give identical tau.
constexpr int ZM_TX = 64, ZM_TY = 8;
constexpr int ZM_HX = ZM_TX + 2, ZM_HP = ZM_HX * (ZM_TY + 2), ZM_NT = ZM_TX * ZM_TY;
constexpr int ZM_PER = (ZM_HP + ZM_NT - 1) / ZM_NT;  // plane nodes per thread

// the plane nodes one thread moves, NC fields each (consecutive fields of `mac` from field F0)
template <typename T, int NC> struct ZmPlane {
    T v[ZM_PER][NC];
};

template <typename T, int NC, int F0>
__device__ __forceinline__ ZmPlane<T, NC> zm_fetch(const Grid& G, const T* __restrict__ mac, int x0, int y0, int zg,
                                                   bool small) {
    ZmPlane<T, NC> r;
    const int64_t zoff = (int64_t)G.px * G.ny * wrap_any(zg, G.nz, small);
#pragma unroll
    for (int i = 0; i < ZM_PER; i++) {
        // unconditional loads (index clamped into the plane) keep the wait a straight count
        const int h0 = threadIdx.x + i * ZM_NT, h = h0 < ZM_HP ? h0 : ZM_HP - 1;
        const int64_t g = wrap_any(x0 + h % ZM_HX - 1, G.nx, small) +
                          (int64_t)G.px * wrap_any(y0 + h / ZM_HX - 1, G.ny, small) + zoff;
#pragma unroll
        for (int k = 0; k < NC; k++) r.v[i][k] = mac[(F0 + k) * G.ns + g];
    }
    return r;
}

template <typename T, int NC> __device__ __forceinline__ void zm_store(const ZmPlane<T, NC>& r, T (*dst)[ZM_HP]) {
#pragma unroll
    for (int i = 0; i < ZM_PER; i++) {
        const int h = threadIdx.x + i * ZM_NT;
        if (h < ZM_HP)
#pragma unroll
            for (int k = 0; k < NC; k++) dst[k][h] = r.v[i][k];
    }
}

__global__ __launch_bounds__(ZM_NT) void les_tau_fp64_zm(Grid G, Phys P, const double* __restrict__ mac,
                                                          const uint64_t* __restrict__ range, int slot,
                                                          double* __restrict__ tau, int tiles_x, int tiles_y, int zc) {
    __shared__ double su[3][3][ZM_HP];  // [ring slot][component][plane node]
    const int x0 = (blockIdx.x % tiles_x) * ZM_TX, y0 = ((blockIdx.x / tiles_x) % tiles_y) * ZM_TY;
    const int zs = (blockIdx.x / (tiles_x * tiles_y)) * zc, ze = min(zs + zc, G.nz);
    const bool small = G.nx <= ZM_TX || G.ny <= ZM_TY || G.nz <= 2;
    const int tx = threadIdx.x % ZM_TX, ty = threadIdx.x / ZM_TX;
    const int x = x0 + tx, y = y0 + ty;
    const bool in = x < G.nx && y < G.ny;
    uint64_t mx_bits, mn_bits;
    range_words(range, slot, mx_bits, mn_bits);
    const double rmax = from_ordered_bits(mx_bits), rmin = from_ordered_bits(mn_bits);
    const double rg = rmax - rmin;
    // ring slot of plane z' is (z' - zs + 1) mod 3
    const auto p0 = zm_fetch<double, 3, 2>(G, mac, x0, y0, zs - 1, small);
    const auto p1 = zm_fetch<double, 3, 2>(G, mac, x0, y0, zs, small);
    const auto p2 = zm_fetch<double, 3, 2>(G, mac, x0, y0, zs + 1, small);
    zm_store(p0, su[0]);
    zm_store(p1, su[1]);
    zm_store(p2, su[2]);
    const int64_t col = G.node(in ? x : 0, in ? y : 0, 0), nxy = (int64_t)G.px * G.ny;
    double phi_next = mac[col + nxy * zs];
    for (int z = zs; z < ze; z++) {
        const bool more = z + 1 < ze;  // plane z+2 is needed by plane z+1
        ZmPlane<double, 3> next;
        if (more) next = zm_fetch<double, 3, 2>(G, mac, x0, y0, z + 2, small);
        const double phi = phi_next;
        if (more) phi_next = mac[col + nxy * (z + 1)];
        __syncthreads();
        if (in) {
            const int rz[3] = {(z - zs) % 3, (z - zs + 1) % 3, (z - zs + 2) % 3};  // planes z-1, z, z+1
            double gu[3][3];
            for (int k = 0; k < 3; k++)
                for (int a = 0; a < 3; a++) gu[k][a] = 0.0;
            sfor<1, 15>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                using D = Dir<q>;
                const int h = (tx + 1 + D::cx) + ZM_HX * (ty + 1 + D::cy);
                for (int k = 0; k < 3; k++) {
                    const double v = su[rz[1 + D::cz]][k][h];
                    gu[k][0] = acc<D::cx>(gu[k][0], v);
                    gu[k][1] = acc<D::cy>(gu[k][1], v);
                    gu[k][2] = acc<D::cz>(gu[k][2], v);
                }
            });
            for (int k = 0; k < 3; k++)
                for (int a = 0; a < 3; a++) gu[k][a] = div_const(gu[k][a], 10.0, 0.1);
            double sum = 0.0;
            for (int b = 0; b < 3; b++)
                for (int a = 0; a < 3; a++) {
                    const double sab = 0.5 * (gu[a][b] + gu[b][a]);
                    sum = sum + sab * sab;
                }
            const double nue = P.les_c * sqrt(2.0 * sum);
            double frac = (phi - rmin) / rg;
            if (rg == 0.0) frac = 0.0;
            const double nu = frac * P.dnu + P.nu1;
            tau[col + nxy * z] = 0.5 + 3.0 * (nu + nue);
        }
        __syncthreads();
        if (more) zm_store(next, su[(z - zs) % 3]);  // the slot of plane z-1
    }
}

// s + v with the rounding error collected in c (TwoSum, Knuth)
__device__ __forceinline__ void add_comp(double& s, double& c, double v) {
    const double t = s + v, b = t - s;
    c += (s - (t - b)) + (v - b);
    s = t;
}

// Diagnostics: per-workgroup partial sums.
// [0] sum phi  [1] sum 0.5|u|^2  [2] sum (d_a u_b + d_b u_a)^2  [3] sum |grad phi|
// [4] sum psi(phi)  [5] sum p  [6..8] sum u  [9] sum_ab d_a phi d_b phi S_ab
// The 40 B per node it must read take 0.11 ms at 256^3; gathering the 56
// neighbour values of every node through L2 took 0.69 ms (this kernel 0.44, bound by
// its 56 LDS reads and about 350 FP64 instructions per node), and 65536 records summed
// on the host another 0.6 ms.  So the workgroups
// march in z like les_tau_fp64_zm, with phi, u of three planes in an LDS ring and
// the next plane's loads in flight, over columns of zc planes; at most
// REDUCE_MAX_BLOCKS of them run, each over a fixed set of columns, and leave one
// record each.  Per-thread sums are compensated, so the longer per-thread chain
// costs no accuracy against the tree over single nodes.
__global__ __launch_bounds__(ZM_NT) void reduce_fp64(Grid G, Phys P, const double* __restrict__ mac,
                                                     double* __restrict__ partial, int tiles_x, int tiles_y, int zc,
                                                     int64_t items) {
    __shared__ double su[3][4][ZM_HP];  // [ring slot][phi, u1, u2, u3][plane node]
    __shared__ double sh[NPART][ZM_NT / 64];
    const int64_t N = G.ns, nxy = (int64_t)G.px * G.ny;
    const bool small = G.nx <= ZM_TX || G.ny <= ZM_TY || G.nz <= 2;
    const int tx = threadIdx.x % ZM_TX, ty = threadIdx.x / ZM_TX;
    double s[NPART] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0}, comp[NPART] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    auto plane = [&](int x0, int y0, int zg) {
        // phi is field 0, u fields 2..4: two fetches of consecutive fields
        ZmPlane<double, 4> r;
        const ZmPlane<double, 1> a = zm_fetch<double, 1, 0>(G, mac, x0, y0, zg, small);
        const ZmPlane<double, 3> b = zm_fetch<double, 3, 2>(G, mac, x0, y0, zg, small);
#pragma unroll
        for (int i = 0; i < ZM_PER; i++) {
            r.v[i][0] = a.v[i][0];
#pragma unroll
            for (int k = 0; k < 3; k++) r.v[i][1 + k] = b.v[i][k];
        }
        return r;
    };
    for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
        const int x0 = (int)(item % tiles_x) * ZM_TX, y0 = (int)((item / tiles_x) % tiles_y) * ZM_TY;
        const int zs = (int)(item / ((int64_t)tiles_x * tiles_y)) * zc, ze = min(zs + zc, G.nz);
        const int x = x0 + tx, y = y0 + ty;
        const bool in = x < G.nx && y < G.ny;
        __syncthreads();  // the ring of the previous column is read no more
        zm_store(plane(x0, y0, zs - 1), su[0]);
        zm_store(plane(x0, y0, zs), su[1]);
        zm_store(plane(x0, y0, zs + 1), su[2]);
        const int64_t col = G.node(in ? x : 0, in ? y : 0, 0);
        double p_next = mac[N + col + nxy * zs];
        int r0 = 0, r1 = 1, r2 = 2;  // ring slots of planes z-1, z, z+1
        for (int z = zs; z < ze; z++) {
            const bool more = z + 1 < ze;  // plane z+2 is needed by plane z+1
            ZmPlane<double, 4> next;
            if (more) next = plane(x0, y0, z + 2);
            const double pr = p_next;
            if (more) p_next = mac[N + col + nxy * (z + 1)];
            __syncthreads();
            if (in) {
                const int rz[3] = {r0, r1, r2};
                const int hc = (tx + 1) + ZM_HX * (ty + 1);
                const double ph = su[r1][0][hc], u1 = su[r1][1][hc], u2 = su[r1][2][hc], u3 = su[r1][3][hc];
                double gp[3] = {0.0, 0.0, 0.0}, gu[3][3];
                for (int k = 0; k < 3; k++)
                    for (int a = 0; a < 3; a++) gu[k][a] = 0.0;
                sfor<1, 15>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    using D = Dir<q>;
                    const int h = hc + D::cx + ZM_HX * D::cy;
                    const double v = su[rz[1 + D::cz]][0][h];
                    gp[0] = acc<D::cx>(gp[0], v);
                    gp[1] = acc<D::cy>(gp[1], v);
                    gp[2] = acc<D::cz>(gp[2], v);
                    for (int k = 0; k < 3; k++) {
                        const double w = su[rz[1 + D::cz]][1 + k][h];
                        gu[k][0] = acc<D::cx>(gu[k][0], w);
                        gu[k][1] = acc<D::cy>(gu[k][1], w);
                        gu[k][2] = acc<D::cz>(gu[k][2], w);
                    }
                });
                for (int a = 0; a < 3; a++) {
                    gp[a] = div_const(gp[a], 10.0, 0.1);
                    for (int k = 0; k < 3; k++) gu[k][a] = div_const(gu[k][a], 10.0, 0.1);
                }
                // interface-strain interaction, ref drop_analysis.f90 korteweg_cal /
                // strain_cal / interaction_cal (:830-882): beta outer, alpha inner
                double e = 0.0, it = 0.0;
                for (int b = 0; b < 3; b++)
                    for (int a = 0; a < 3; a++) {
                        const double sab = gu[a][b] + gu[b][a];
                        e += sab * sab;
                        it = it + (gp[a] * gp[b]) * (0.5 * sab);
                    }
                add_comp(s[0], comp[0], ph);
                add_comp(s[1], comp[1], 0.5 * (u1 * u1 + u2 * u2 + u3 * u3));
                add_comp(s[2], comp[2], e);
                add_comp(s[3], comp[3], sqrt(gp[0] * gp[0] + gp[1] * gp[1] + gp[2] * gp[2]));
                add_comp(s[4], comp[4], ph * P.T * log(ph / (1.0 - P.b * ph)) - P.a * ph * ph);
                add_comp(s[5], comp[5], pr);
                add_comp(s[6], comp[6], u1);
                add_comp(s[7], comp[7], u2);
                add_comp(s[8], comp[8], u3);
                add_comp(s[9], comp[9], it);
            }
            __syncthreads();
            if (more) zm_store(next, su[r0]);  // the slot of plane z-1
            const int t = r0;
            r0 = r1;
            r1 = r2;
            r2 = t;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = 0; k < NPART; k++) {
        double t = s[k] + comp[k];
        for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
        if (lane == 0) sh[k][wave] = t;
    }
    __syncthreads();
    if (threadIdx.x < NPART) {
        const int k = threadIdx.x;
        double t = sh[k][0];
        for (int w = 1; w < ZM_NT / 64; w++) t += sh[k][w];
        partial[(int64_t)blockIdx.x * NPART + k] = t;
    }
}

// Compensated sums of the workgroups' records (fixed order: lane l of wavefront k
// takes records l, l + 64, ... of component k, then a tree over the lanes), and the
// phi range next to them, so that one small copy returns everything.
__global__ __launch_bounds__(64 * NPART) void reduce_final(const double* __restrict__ partial, int nblocks,
                                                           const uint64_t* __restrict__ range, int slot,
                                                           double* __restrict__ out) {
    const int lane = threadIdx.x & 63, k = threadIdx.x >> 6;
    double s = 0.0, c = 0.0;
#pragma unroll 4
    for (int b = lane; b < nblocks; b += 64) add_comp(s, c, partial[(int64_t)b * NPART + k]);
    for (int off = 32; off > 0; off >>= 1) {
        const double so = __shfl_xor(s, off, 64), co = __shfl_xor(c, off, 64);
        add_comp(s, c, so);
        c += co;
    }
    if (lane == 0) out[k] = s + c;
    if (threadIdx.x == 0) {
        uint64_t* const words = reinterpret_cast<uint64_t*>(out + NPART);
        range_words(range, slot, words[0], words[1]);
    }
}

// rows of nx doubles, `stride` apart, to contiguous rows; one thread per value
__global__ __launch_bounds__(256) void pack_rows(int nx, int64_t rows, int64_t stride, const double* __restrict__ nodes,
                                                 double* __restrict__ packed) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t row = i / nx;
    if (row < rows) packed[i] = nodes[(i - row * nx) + stride * row];
}

__global__ void range_set(uint64_t* range, int slot, double vmax, double vmin) {
    range_set_part(range, slot, threadIdx.x, ordered_bits(vmax), ordered_bits(vmin));
}

// ------------------------------------------------------------------ launchers
static inline int64_t nblk(int64_t n, int bs) { return (n + bs - 1) / bs; }

hipError_t launch_init_equilibrium_fp64(const Grid& G, const Phys& ph, const double* mac, double* f,
                                        double* g, hipStream_t st) {
    hipLaunchKernelGGL(init_equilibrium_fp64, dim3(nblk(G.slots(), 256)), dim3(256), 0, st, G, ph, mac, f, g);
    return hipGetLastError();
}

hipError_t launch_moments_fp64(const Grid& G, const double* f, const double* g, double* mac, int which,
                               hipStream_t st) {
    hipLaunchKernelGGL(moments_fp64, dim3(nblk(G.slots(), 256)), dim3(256), 0, st, G, f, g, mac, which);
    return hipGetLastError();
}

hipError_t launch_les_tau_fp64(const Grid& G, const Phys& ph, const double* mac, const double* mac_old,
                               const LesBlocks& blk, const uint64_t* range, int slot, double* tau, hipStream_t st) {
    const int tx = (G.nx + LES_TX - 1) / LES_TX, ty = (G.ny + LES_TY - 1) / LES_TY, tz = (G.nz + LES_TZ - 1) / LES_TZ;
    const dim3 grid((unsigned)(tx * ty * tz)), block(LES_TX * LES_TY * LES_TZ);
    if (blk.bx > 0 && mac_old != mac) {
        hipLaunchKernelGGL(les_tau_fp64<true>, grid, block, 0, st, G, ph, mac, mac_old, blk, range, slot, tau, tx, ty);
    } else {
        const int mx = (G.nx + ZM_TX - 1) / ZM_TX, my = (G.ny + ZM_TY - 1) / ZM_TY;
        const int zc = les_planes(mx * my, G.nz), mz = (G.nz + zc - 1) / zc;
        hipLaunchKernelGGL(les_tau_fp64_zm, dim3((unsigned)(mx * my * mz)), dim3(ZM_TX * ZM_TY), 0, st, G, ph, mac, range,
                           slot, tau, mx, my, zc);
    }
    return hipGetLastError();
}

hipError_t launch_reduce_fp64(const Grid& G, const Phys& ph, const double* mac, const uint64_t* range, int slot,
                              double* work, hipStream_t st) {
    const int mx = (G.nx + ZM_TX - 1) / ZM_TX, my = (G.ny + ZM_TY - 1) / ZM_TY;
    // columns of up to 32 planes (the two halo planes cost 2 / zc), shorter where the
    // lattice would leave less than four workgroups per CU
    const int64_t planes = (int64_t)mx * my * G.nz;
    const int zc = (int)std::min<int64_t>(std::min(32, G.nz), std::max<int64_t>(1, planes / 1024));
    const int64_t items = (int64_t)mx * my * ((G.nz + zc - 1) / zc);
    const int nblocks = (int)std::min<int64_t>(items, REDUCE_MAX_BLOCKS);
    hipLaunchKernelGGL(reduce_fp64, dim3(nblocks), dim3(ZM_NT), 0, st, G, ph, mac, work, mx, my, zc, items);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(reduce_final, dim3(1), dim3(64 * NPART), 0, st, (const double*)work, nblocks, range, slot,
                       work + REDUCE_OUT);
    return hipGetLastError();
}

hipError_t launch_pack_rows(int nx, int64_t rows, int64_t stride, const double* nodes, double* packed, hipStream_t st) {
    hipLaunchKernelGGL(pack_rows, dim3(nblk(nx * rows, 256)), dim3(256), 0, st, nx, rows, stride, nodes, packed);
    return hipGetLastError();
}

hipError_t launch_range_set(uint64_t* range, int slot, double vmax, double vmin, hipStream_t st) {
    hipLaunchKernelGGL(range_set, dim3(1), dim3(RANGE_PARTS), 0, st, range, slot, vmax, vmin);
    return hipGetLastError();
}

}  // namespace drp
