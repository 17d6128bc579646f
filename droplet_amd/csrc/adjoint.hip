// adjoint.hip — discrete adjoint of the FP64 two-phase step (reverse mode, by hand).
//
// Forward step n -> n+1 (step_kernels.hip): at every node y the equilibria
// feq(phi, p0, lap phi, grad phi, u) and geq(p, u, grad phi) are formed from the
// stored macroscopic fields m^n = (phi, p, u), the populations relax
//   f*_q(y) = f_q(y) - (f_q(y) - feq_q(y)) / tau_f,
//   g*_q(y) = g_q(y) - (g_q(y) - geq_q(y)) / tau_g + force,
// stream to y + c_q, the momentum populations entering the fluid on a wall
// layer are overwritten by bounce-back, and m^{n+1} = moments(f^{n+1}, g^{n+1}).
//
// With Fh, Gh the adjoints of f^{n+1}, g^{n+1} (total: they include the use
// of m^{n+1} in the next step), one reverse step is
//   kernel A (per node y, pulling from y + c_q):
//     Fh*_q(y) = Fh_q(y + c_q),  Gh*_q(y) = bounce-back transpose of Gh at y + c_q;
//     adjoints of feq / geq = Fh* / tau_f, Gh* / tau_g  ->  local adjoints of
//     phi, p, u, the F-bracket A, lap phi and grad phi at y;
//     Fh^n_q(y) = (1 - 1/tau_f) Fh*_q(y) + phih_local(y)      (stencil part below)
//     Gh^n_q(y) = (1 - 1/tau_g) Gh*_q(y) + ph(y)/3 + c_q . uh(y)
//     parameter sensitivities  d/dtau_f, d/dkappa_g, d/dU_wall  (per workgroup)
//   kernel B (per node x): the transposed lap / grad stencil
//     phih_st(x) = -14/5 laph(x) + sum_q [laph(x - c_q)/5 + c_q . gradh(x - c_q)/10]
// and the next reverse step reads Fh^n_q(x) = Fpart_q(x) + phih_st(x).
//
// Restrictions (checked on the host): equal viscosities (tau_g constant, so the
// global phi range never enters), no Smagorinsky model.  Body forces are
// additive and state independent and so drop out of the adjoint.
#include <climits>
#include <type_traits>
#include <utility>

#include "d3q15.h"
#include "kernels.h"

namespace drp {

namespace {
constexpr int CX[15] = {0, 1, 0, 0, -1, 0, 0, 1, -1, 1, 1, -1, 1, -1, -1};
constexpr int CY[15] = {0, 0, 1, 0, 0, -1, 0, 1, 1, -1, 1, -1, -1, 1, -1};
constexpr int CZ[15] = {0, 0, 0, 1, 0, 0, -1, 1, 1, 1, -1, -1, -1, -1, 1};
constexpr int OPP[15] = {0, 4, 5, 6, 1, 2, 3, 11, 12, 13, 14, 7, 8, 9, 10};
constexpr double EW[15] = {2.0 / 9.0, 1.0 / 9.0, 1.0 / 9.0, 1.0 / 9.0, 1.0 / 9.0, 1.0 / 9.0, 1.0 / 9.0,
                           1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0, 1.0 / 72.0,
                           1.0 / 72.0};
constexpr double FW[15] = {-7.0 / 3.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 3.0, 1.0 / 3.0,
                           1.0 / 24.0, 1.0 / 24.0, 1.0 / 24.0, 1.0 / 24.0, 1.0 / 24.0, 1.0 / 24.0, 1.0 / 24.0,
                           1.0 / 24.0};
constexpr int ADJ_BLOCK = 256;

__device__ __forceinline__ int wrap1(int v, int n) { return v < 0 ? v + n : (v >= n ? v - n : v); }

// node coordinates and indices in 32 bits: the tape admits fewer than 2^32 nodes,
// row padding included
struct Node {
    int x, y, z;
};
__device__ __forceinline__ Node coords(uint32_t s, const Grid& G) {
    const uint32_t nxy = (uint32_t)G.px * (uint32_t)G.ny;
    Node c;
    c.z = (int)(s / nxy);
    const uint32_t r = s - (uint32_t)c.z * nxy;
    c.y = (int)(r / (uint32_t)G.px);
    c.x = (int)(r - (uint32_t)c.y * (uint32_t)G.px);
    return c;
}
__device__ __forceinline__ uint32_t shifted(const Node& c, int dx, int dy, int dz, const Grid& G) {
    return (uint32_t)wrap1(c.x + dx, G.nx) +
           (uint32_t)G.px * ((uint32_t)wrap1(c.y + dy, G.ny) + (uint32_t)G.ny * (uint32_t)wrap1(c.z + dz, G.nz));
}

// workgroup sum of three partials, added into acc[0..2], the tile's own (so the
// accumulation order is fixed)
__device__ void block_accumulate(double v0, double v1, double v2, double* acc) {
    __shared__ double sh[3][ADJ_BLOCK / 64];
    double v[3] = {v0, v1, v2};
#pragma unroll
    for (int k = 0; k < 3; k++)
        for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0)
        for (int k = 0; k < 3; k++) sh[k][wave] = v[k];
    __syncthreads();
    if (threadIdx.x < 3) {
        double t = sh[threadIdx.x][0];
        for (int w = 1; w < ADJ_BLOCK / 64; w++) t += sh[threadIdx.x][w];
        acc[threadIdx.x] += t;
    }
}
}  // namespace

template <int Q>
using Vel = std::integral_constant<int, Q>;
template <int... Q, class F>
__device__ __forceinline__ void each_dir(std::integer_sequence<int, Q...>, F&& f) {
    (f(Vel<Q>{}), ...);
}
// f(Vel<q>) for q = 0 .. 14
template <class F>
__device__ __forceinline__ void all_dirs(F&& f) {
    each_dir(std::make_integer_sequence<int, 15>{}, f);
}
// c_q . v, without the products by zero
template <int Q>
__device__ __forceinline__ double cdot(const double (&v)[3]) {
    double t = 0.0;
    if constexpr (CX[Q] != 0) t += CX[Q] * v[0];
    if constexpr (CY[Q] != 0) t += CY[Q] * v[1];
    if constexpr (CZ[Q] != 0) t += CZ[Q] * v[2];
    return t;
}

// sums over the directions with the weights E: 1 (without the rest direction), c_k and
// c_k c_l (xx, yy, zz, xy, xz, yz)
struct Moments {
    double s, p[3], t[6];
};
__device__ __forceinline__ Moments moments(const double (&v)[15]) {
    Moments m;
    double c0 = 0.0, c1[3] = {0.0, 0.0, 0.0}, c2[3] = {0.0, 0.0, 0.0};
    all_dirs([&](auto d) {
        constexpr int q = d;
        if constexpr (q >= 7) {
            c0 += v[q];
            c1[0] += CX[q] * v[q];
            c1[1] += CY[q] * v[q];
            c1[2] += CZ[q] * v[q];
            c2[0] += CX[q] * CY[q] * v[q];
            c2[1] += CX[q] * CZ[q] * v[q];
            c2[2] += CY[q] * CZ[q] * v[q];
        }
    });
    m.s = EW[7] * c0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double pair = EW[1] * (v[1 + k] + v[4 + k]);
        m.s += pair;
        m.p[k] = EW[1] * (v[1 + k] - v[4 + k]) + EW[7] * c1[k];
        m.t[k] = pair + EW[7] * c0;
        m.t[3 + k] = EW[7] * c2[k];
    }
    return m;
}
// r = t v, t symmetric as in Moments
__device__ __forceinline__ void mul(const double (&t)[6], const double (&v)[3], double (&r)[3]) {
    r[0] = t[0] * v[0] + t[3] * v[1] + t[4] * v[2];
    r[1] = t[3] * v[0] + t[1] * v[1] + t[5] * v[2];
    r[2] = t[4] * v[0] + t[5] * v[1] + t[2] * v[2];
}

// One pass over 15 f, 30 adjoint populations in and 30 out: bound by HBM, 85 values a
// node with the fields and the gradients out.  Kept at 64 bits and read once, the 30 take
// 60 VGPRs, so three wavefronts per SIMD (162 VGPRs, 45 loads in flight in each).  With
// rolled loops over the directions, five wavefronts and the 30 read a second time for the
// outputs the second read came from beyond the L2: 200 us at 96^3, 124 now (the bytes take
// 106).  The per-direction sums of the outputs (uh, gh, Ah) taken in 15 terms each kept
// their factors alive to the end and spilled; from the moments of the 30 they do not.
// Workgroups in XCD order: phi and phih_st are read at 15 nodes each, from one L2 then.
template <int WALL, bool FIRST>
__global__ __launch_bounds__(ADJ_BLOCK) __attribute__((amdgpu_waves_per_eu(3))) void adj_collide_fp64(AdjArgs a) {
    const Grid& G = a.G;
    const int64_t n = G.ns;  // from one array to the next
    const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
    const uint32_t s = tile * (uint32_t)ADJ_BLOCK + threadIdx.x;
    double d_tauf = 0.0, d_kg = 0.0, d_u = 0.0;
    const Node c = coords(s, G);
    if (c.x < G.nx && s < (uint64_t)G.slots()) {
        // adjoints entering the post-collision populations of y, i.e. those of
        // the streamed populations at the downstream node d = y + c_q
        uint32_t down[15];
        double Fs[15], Gs[15];
        all_dirs([&](auto d) {
            constexpr int q = d;
            down[q] = shifted(c, CX[q], CY[q], CZ[q], G);
            Fs[q] = a.Fin[q * n + down[q]];
            Gs[q] = a.Gin[q * n + down[q]];
        });
        // forward stencils at y (various_cal)
        const double phi = a.mac[s];
        const double u[3] = {a.mac[2 * n + s], a.mac[3 * n + s], a.mac[4 * n + s]};
        double lap = -14.0 * phi, gr[3] = {0.0, 0.0, 0.0};
        all_dirs([&](auto d) {
            constexpr int q = d;
            Fs[q] += a.phin_in[down[q]];
            if constexpr (q > 0) {
                const double v = a.mac[down[q]];
                lap += v;
                if constexpr (CX[q] != 0) gr[0] += CX[q] * v;
                if constexpr (CY[q] != 0) gr[1] += CY[q] * v;
                if constexpr (CZ[q] != 0) gr[2] += CZ[q] * v;
            }
        });
        // bounce-back transpose on wall layers
        const int w = (WALL == 2) ? c.y : c.z, wn = (WALL == 2) ? G.ny : G.nz;
        if constexpr (WALL != 0) {
            if (w <= 1 || w >= wn - 2)
                all_dirs([&](auto d) {
                    constexpr int q = d;
                    constexpr int ca = (WALL == 2) ? CY[q] : CZ[q];
                    if constexpr (ca != 0) {
                        if (w == (ca > 0 ? wn - 1 : 0)) Gs[q] = 0.0;       // overwritten at d
                        else if (w == (ca > 0 ? wn - 2 : 1)) Gs[q] += a.Gin[OPP[q] * n + down[q]];  // copied into opp(q) at d
                    }
                });
        }
        lap /= 5.0;
        gr[0] /= 10.0;
        gr[1] /= 10.0;
        gr[2] /= 10.0;
        const double gsq = gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2];
        const double ombp = 1.0 - a.b * phi;
        const double p0 = phi * a.T / ombp - a.a * phi * phi;
        const double A = p0 - a.kf * phi * lap - a.kf6 * gsq;

        // Fs . (f - feq), direction by direction: the difference is small against both
        all_dirs([&](auto d) {
            constexpr int q = d;
            constexpr double c2 = (double)(CX[q] * CX[q] + CY[q] * CY[q] + CZ[q] * CZ[q]);
            double fe = FW[q] * A;
            if constexpr (q == 0) {
                fe += phi;
            } else {
                const double cg = cdot<q>(gr);
                fe += 3.0 * EW[q] * phi * cdot<q>(u) + EW[q] * a.kf * (4.5 * cg * cg - 1.5 * gsq * c2);
            }
            d_tauf += Fs[q] * (a.f[q * n + s] - fe);
        });
        d_tauf *= a.rtau_f2;
        // the adjoints of feq and geq are Fs / tau_f and Gs / tau_g; feq and geq are linear in
        // their fields with c, c c and 1 as coefficients, so the moments of Fs and Gs suffice
        const Moments mf = moments(Fs), mg = moments(Gs);
        const double Ah = a.rtau_f * (FW[0] * Fs[0] + 3.0 * mf.s);
        const double g0 = mg.s + EW[0] * Gs[0];
        const double ph = 3.0 * a.rtau_g * g0;
        const double dp0 = a.T / (ombp * ombp) - 2.0 * a.a * phi;
        const double phih = a.rtau_f * (Fs[0] + 3.0 * (mf.p[0] * u[0] + mf.p[1] * u[1] + mf.p[2] * u[2])) +
                            Ah * (dp0 - a.kf * lap);
        const double laph = -a.kf * phi * Ah;
        double uh[3], gh[3], qu[3], qg[3], wg[3];
        mul(mg.t, u, qu);
        mul(mg.t, gr, qg);
        const double kff = a.kf * a.rtau_f, kgg = a.kg * a.rtau_g;
        double w2[6];
#pragma unroll
        for (int k = 0; k < 6; k++) w2[k] = kff * mf.t[k] + kgg * mg.t[k];
        mul(w2, gr, wg);
        const double trw = w2[0] + w2[1] + w2[2];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            uh[k] = 3.0 * phi * a.rtau_f * mf.p[k] + a.rtau_g * (3.0 * mg.p[k] + 9.0 * qu[k] - 3.0 * u[k] * g0);
            gh[k] = 9.0 * wg[k] - 3.0 * gr[k] * trw - 2.0 * a.kf6 * gr[k] * Ah;
        }
        // Gs . (E times the kappa_g part of geq)
        const double kg1 = 4.5 * (gr[0] * qg[0] + gr[1] * qg[1] + gr[2] * qg[2]) -
                           1.5 * gsq * (mg.t[0] + mg.t[1] + mg.t[2]);
        // populations of an initial state are geq / feq of constant fields:
        // only the kappa_g dependence of g^0 = geq(m^0) remains
        d_kg = (FIRST ? a.rtau_g + a.om_g : a.rtau_g) * kg1;

        const double p3 = ph / 3.0;
        all_dirs([&](auto d) {
            constexpr int q = d;
            const double Fp = a.om_f * Fs[q], Gp = a.om_g * Gs[q];
            if constexpr (FIRST) {
                a.Fout[q * n + s] = Fp;
                a.Gout[q * n + s] = Gp;
            } else {
                a.Fout[q * n + s] = Fp + phih;
                a.Gout[q * n + s] = Gp + p3 + cdot<q>(uh);
            }
        });
        if constexpr (!FIRST) {
            a.lapA[s] = laph;
            a.gradA[s] = gh[0];
            a.gradA[n + s] = gh[1];
            a.gradA[2 * n + s] = gh[2];
        }

        // wall speed: on a wall layer g_j = g_opp(j) - 6 E_opp (U_w . c_opp), U_w = (-+U, 0, 0)
        if constexpr (WALL != 0) {
            const bool bottom = w == 0, top = w == wn - 1;
            if (a.wall_active && (bottom || top)) {
                const int want = bottom ? 1 : -1;
                const double sgn = bottom ? -1.0 : 1.0;
                all_dirs([&](auto d) {
                    constexpr int q = d;
                    constexpr int ca = (WALL == 2) ? CY[q] : CZ[q];
                    constexpr int o = OPP[q];
                    if constexpr (ca != 0 && CX[o] != 0)
                        if (ca == want) d_u += a.Gin[q * n + s] * (-6.0 * EW[o] * (double)CX[o] * sgn);
                });
            }
        }
    }
    block_accumulate(d_tauf, d_kg, d_u, a.acc + 3 * (int64_t)tile);
}

// phih_st(x) = -14/5 laph(x) + sum_{q>=1} [laph(x - c_q)/5 + c_q . gradh(x - c_q)/10]
// 57 values are read for each node.  From memory they bound it: 29 us at 96^3, where
// the four arrays and the result take 6.  Tiles of the four arrays with their halos in
// LDS: 15 us; 2.4 nodes are staged for each of a tile.
constexpr int ST_X = 32, ST_Y = 4, ST_Z = 4, ST_BLOCK = ST_X * ST_Y * ST_Z;
constexpr int ST_HX = ST_X + 2, ST_HY = ST_Y + 2, ST_HN = ST_HX * ST_HY * (ST_Z + 2);
__global__ __launch_bounds__(ST_BLOCK) void adj_stencil_fp64(Grid G, int tiles_x, int tiles_y, int tiles,
                                                             const double* __restrict__ lapA,
                                                             const double* __restrict__ gradA,
                                                             double* __restrict__ out) {
    __shared__ double v[4][ST_HN];
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= tiles) return;
    const int x0 = tile % tiles_x * ST_X, y0 = tile / tiles_x % tiles_y * ST_Y, z0 = tile / (tiles_x * tiles_y) * ST_Z;
    const int64_t n = G.ns;
    for (int i = threadIdx.x; i < ST_HN; i += ST_BLOCK) {
        const int x = x0 - 1 + i % ST_HX, y = y0 - 1 + i / ST_HX % ST_HY, z = z0 - 1 + i / (ST_HX * ST_HY);
        // one layer beyond the lattice is its halo; what lies further out has no reader
        if (x <= G.nx && y <= G.ny && z <= G.nz) {
            const int64_t s = G.at(x, y, z);
            v[0][i] = lapA[s];
            v[1][i] = gradA[s];
            v[2][i] = gradA[n + s];
            v[3][i] = gradA[2 * n + s];
        }
    }
    __syncthreads();
    const int lx = threadIdx.x % ST_X, ly = threadIdx.x / ST_X % ST_Y, lz = threadIdx.x / (ST_X * ST_Y);
    if (x0 + lx >= G.nx || y0 + ly >= G.ny || z0 + lz >= G.nz) return;
    const int h = lx + 1 + ST_HX * (ly + 1 + ST_HY * (lz + 1));
    double l = 0.0, g = 0.0;
    all_dirs([&](auto d) {
        constexpr int q = d;
        if constexpr (q > 0) {
            constexpr int off = CX[q] + ST_HX * (CY[q] + ST_HY * CZ[q]);
            const double gq[3] = {v[1][h - off], v[2][h - off], v[3][h - off]};
            l += v[0][h - off];
            g += cdot<q>(gq);
        }
    });
    out[G.node(x0 + lx, y0 + ly, z0 + lz)] = -14.0 / 5.0 * v[0][h] + l / 5.0 + g / 10.0;
}

// seed of sum_x |grad phi(x)|: gradA = w grad phi / |grad phi| (0 where grad phi = 0), lapA = 0
__global__ __launch_bounds__(ADJ_BLOCK) void adj_seed_area_fp64(Grid G, const double* __restrict__ phi,
                                                                double w, double* __restrict__ lapA,
                                                                double* __restrict__ gradA) {
    const uint32_t s = blockIdx.x * (uint32_t)ADJ_BLOCK + threadIdx.x;
    const Node c = coords(s, G);
    if (c.x >= G.nx || s >= (uint64_t)G.slots()) return;
    const int64_t n = G.ns;
    double gr[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 1; q < 15; q++) {
        const double v = phi[shifted(c, CX[q], CY[q], CZ[q], G)];
        gr[0] += CX[q] * v;
        gr[1] += CY[q] * v;
        gr[2] += CZ[q] * v;
    }
    const double m = sqrt(gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2]);  // 10 |grad phi|
    const double sc = m > 0.0 ? w / m : 0.0;
    lapA[s] = 0.0;
    gradA[s] = gr[0] * sc;
    gradA[n + s] = gr[1] * sc;
    gradA[2 * n + s] = gr[2] * sc;
}

// out[plane node (i, j)] += vals[j * n1 + i]; the plane is (x, y) at z = third
// (wall_y) or (x, z) at y = third
__global__ void adj_add_plane(Grid G, int n1, int n2, int wall_y, int third, const double* __restrict__ vals,
                              double* __restrict__ out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n1 * n2) return;
    const int i = t % n1, j = t / n1;
    const int64_t s = wall_y ? G.node(i, j, third) : G.node(i, third, j);
    out[s] += vals[t];
}

// ------------------------------------------------------------------ launchers
// a multiple of 8, for xcd_tile; the workgroups beyond the last node only add zeros
static inline int nblocks(int64_t n) { return (int)(((n + ADJ_BLOCK - 1) / ADJ_BLOCK + 7) & ~(int64_t)7); }

int adj_block_count(const Grid& G) { return nblocks(G.slots()); }

hipError_t launch_adj_collide_fp64(const AdjArgs& a, hipStream_t st) {
    auto* k = adj_collide_fp64<0, false>;
    if (a.wall_axis == 0) k = a.first ? adj_collide_fp64<0, true> : adj_collide_fp64<0, false>;
    else if (a.wall_axis == 2) k = a.first ? adj_collide_fp64<2, true> : adj_collide_fp64<2, false>;
    else k = a.first ? adj_collide_fp64<3, true> : adj_collide_fp64<3, false>;
    hipLaunchKernelGGL(k, dim3(nblocks(a.G.slots())), dim3(ADJ_BLOCK), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_adj_stencil_fp64(const Grid& G, const double* lapA, const double* gradA, double* out,
                                   hipStream_t st) {
    const int tx = (G.nx + ST_X - 1) / ST_X, ty = (G.ny + ST_Y - 1) / ST_Y, tz = (G.nz + ST_Z - 1) / ST_Z;
    const int64_t tiles = (int64_t)tx * ty * tz;
    if (tiles > INT_MAX - 7) return hipErrorInvalidValue;
    hipLaunchKernelGGL(adj_stencil_fp64, dim3((uint32_t)(tiles + 7) / 8 * 8), dim3(ST_BLOCK), 0, st, G, tx, ty, (int)tiles,
                       lapA, gradA, out);
    return hipGetLastError();
}

hipError_t launch_adj_seed_area_fp64(const Grid& G, const double* phi, double w, double* lapA,
                                     double* gradA, hipStream_t st) {
    hipLaunchKernelGGL(adj_seed_area_fp64, dim3(nblocks(G.slots())), dim3(ADJ_BLOCK), 0, st, G,
                       phi, w, lapA, gradA);
    return hipGetLastError();
}

hipError_t launch_adj_add_plane(const Grid& G, int n1, int n2, int wall_y, int third, const double* vals,
                                double* out, hipStream_t st) {
    hipLaunchKernelGGL(adj_add_plane, dim3((n1 * n2 + 255) / 256), dim3(256), 0, st, G, n1, n2, wall_y, third,
                       vals, out);
    return hipGetLastError();
}

}  // namespace drp
