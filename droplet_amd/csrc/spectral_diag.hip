// spectral_diag.hip — FFT diagnostics of the velocity field on the GPU:
//
//   drp_energy_spectrum     enesupe_cal, program/turbulence_hit_xy.f90:588-644
//   drp_filter_velocity     low_pass, program/LES_drop_xy.f90:851-971 (keep the
//                           shells int|k| < k) and the band-pass of scale_cal2,
//                           program/drop_analysis.f90:722-797 (keep int|k| == k)
//   drp_scale_interaction   the per-scale interface-velocity interaction of
//                           program/drop_analysis.f90:1121-1265:
//                           C(k) = kappa_g < u^(k) . div(grad phi grad phi) >
//   drp_phi_contribution    the cross spectrum of u . grad phi and the chemical
//                           potential, contribution of drop_analysis.f90:476-578
//
// The reference transforms with 2decomp/FFTW (r2c with the halved axis z,
// u_hat = FFT(u) / (nx ny nz), signed wavenumber k = i - n for i >= n/2 + 1).
// Here a 3-D FFT is one mixed-radix Stockham pass per axis (radices 8, 4, 2, 3, 5;
// every extent a product of those, at most 2048): each workgroup loads G whole
// lines into LDS, runs the log_R(n) stages there with twiddles from a table
// e^{-2 pi i t / n} evaluated on the host, and writes the lines back in place.
// Lines along y and z are taken G at a time with consecutive x, so their loads and
// stores are coalesced.
//
// The spectra transform real fields, so they keep the half spectrum kx = 0..nx/2:
// the x pass packs two real rows into one complex line and separates their
// transforms on the way out, the y pass works on nx/2 + 1 lines per plane, and the
// z pass writes nothing back: its lines go from LDS straight into shell bins.  A
// stored mode stands for itself and for its mirror image -k where that is not
// stored too.  One field is transformed at a time, so its half spectrum (143 MB at
// 256^3) passes from kernel to kernel through the 256 MB last-level cache.
//
// The per-scale interaction uses Parseval instead of one inverse transform per
// shell: < u^(k) . w > = sum over the modes of shell k of Re(u_hat w_hat*), with
// both transforms normalised by the node count; it equals the reference's
// physical-space mean of the band-passed velocity times w up to rounding.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <new>
#include <vector>

#include "../../include/droplet.h"
#include "d3q15.h"
#include "kernels.h"
#include "lattice_impl.h"

using namespace drp;

namespace {

#define HIP_TRYS(expr)                                                                      \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess)                                                               \
            return drp_fail(DRP_ERR_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));    \
    } while (0)

constexpr int FFT_MAX_STAGES = 12;
constexpr int FFT_BLOCK = 256;       // threads per workgroup
constexpr int FFT_MAX_LINE = 2048;   // longest line
// complex numbers of one workgroup's G lines (32 KiB of LDS: five workgroups per CU).
// Eight 256-point lines make the strided passes touch whole 128-byte lines of memory
// (four lines, with a second LDS buffer for the stages, ran at 2.4 TB/s)
constexpr int FFT_POINTS = 2048;

struct FFTAxis {
    int L;                     // line length
    int64_t S;                 // element stride along the line
    int64_t nlines;            // lines of this axis
    int F;                     // lines per row of the fastest other coordinate
    int64_t sf, so;            // base = (l % F) * sf + (l / F) * so
    int G;                     // lines per workgroup
    int nst;                   // stages
    int rad[FFT_MAX_STAGES];   // radix of each stage
    uint32_t mm[FFT_MAX_STAGES], mn[FFT_MAX_STAGES];  // 2^32 / M and 2^32 / Ns of each stage, rounded up
                                                      // (0 for a divisor of 1): quotients by one multiply
    uint32_t ml;               // the same for L
    const double2* tw;         // e^{-2 pi i t / L}, t = 0..L-1
};

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// R-point DFT o[q] = sum_r v[r] W^(r q), W = e^{s 2 pi i / R} (s = -1 forward,
// +1 inverse), with the roots of unity as constants
template <int R> __device__ __forceinline__ void small_dft(const double2 (&v)[R], double2 (&o)[R], int sign) {
    const double s = (double)sign;
    if constexpr (R == 2) {
        o[0] = make_double2(v[0].x + v[1].x, v[0].y + v[1].y);
        o[1] = make_double2(v[0].x - v[1].x, v[0].y - v[1].y);
    } else if constexpr (R == 4) {
        // W = s i: W z = (-s z.y, s z.x)
        const double2 a = make_double2(v[0].x + v[2].x, v[0].y + v[2].y);
        const double2 b = make_double2(v[0].x - v[2].x, v[0].y - v[2].y);
        const double2 c = make_double2(v[1].x + v[3].x, v[1].y + v[3].y);
        const double2 d = make_double2(v[1].x - v[3].x, v[1].y - v[3].y);
        const double2 wd = make_double2(-s * d.y, s * d.x);
        o[0] = make_double2(a.x + c.x, a.y + c.y);
        o[1] = make_double2(b.x + wd.x, b.y + wd.y);
        o[2] = make_double2(a.x - c.x, a.y - c.y);
        o[3] = make_double2(b.x - wd.x, b.y - wd.y);
    } else if constexpr (R == 8) {
        // even and odd 4-point halves, W = (1 + s i) / sqrt 2
        constexpr double H = 0.70710678118654752440;
        const double2 ev[4] = {v[0], v[2], v[4], v[6]}, od[4] = {v[1], v[3], v[5], v[7]};
        double2 e[4], d[4];
        small_dft<4>(ev, e, sign);
        small_dft<4>(od, d, sign);
        const double2 w[4] = {d[0], make_double2(H * (d[1].x - s * d[1].y), H * (d[1].y + s * d[1].x)),
                              make_double2(-s * d[2].y, s * d[2].x),
                              make_double2(-H * (d[3].x + s * d[3].y), H * (s * d[3].x - d[3].y))};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            o[q] = make_double2(e[q].x + w[q].x, e[q].y + w[q].y);
            o[q + 4] = make_double2(e[q].x - w[q].x, e[q].y - w[q].y);
        }
    } else {
        // R = 3, 5: cos and sin of 2 pi m / R
        constexpr double C3[3] = {1.0, -0.5, -0.5};
        constexpr double S3[3] = {0.0, 0.86602540378443864676, -0.86602540378443864676};
        constexpr double C5[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410, -0.80901699437494742410,
                                  0.30901699437494742410};
        constexpr double S5[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917, -0.58778525229247312917,
                                  -0.95105651629515357212};
#pragma unroll
        for (int q = 0; q < R; q++) {
            double2 acc = v[0];
#pragma unroll
            for (int r = 1; r < R; r++) {
                const int m = (r * q) % R;
                const double wc = R == 3 ? C3[m] : C5[m], ws = s * (R == 3 ? S3[m] : S5[m]);
                acc.x += v[r].x * wc - v[r].y * ws;
                acc.y += v[r].x * ws + v[r].y * wc;
            }
            o[q] = acc;
        }
    }
}

// b / d for b < 2^16 from m = ceil(2^32 / d), d < 2^16 (m = 0: d = 1)
__device__ __forceinline__ uint32_t quotient(uint32_t b, uint32_t m) { return m ? __umulhi(b, m) : b; }

// one Stockham stage of radix R, in place, over the ng lines of length L held in
// LDS: every thread reads its butterflies into registers before any is written
template <int R>
__device__ __forceinline__ void fft_stage(double2* buf, const FFTAxis& A, int st, int ng, int Ns, int sign) {
    constexpr int NB = (FFT_POINTS / R + FFT_BLOCK - 1) / FFT_BLOCK;  // butterflies per thread
    const int L = A.L, M = L / R, step = L / (Ns * R), nb = ng * M;
    double2 o[NB][R];
    int to[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const int b = threadIdx.x + i * FFT_BLOCK;
        to[i] = -1;
        if (b >= nb) continue;
        const int g = (int)quotient(b, A.mm[st]), j = b - g * M;
        const int k = j - (int)quotient(j, A.mn[st]) * Ns;
        const double2* sl = buf + g * L;
        double2 v[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            double2 x = sl[j + r * M];
            if (r > 0 && Ns > 1) {
                double2 w = A.tw[k * r * step];  // k r step < L
                if (sign > 0) w.y = -w.y;
                x = cmul(x, w);
            }
            v[r] = x;
        }
        small_dft<R>(v, o[i], sign);
        to[i] = g * L + (j - k) * R + k;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; i++) {
        if (to[i] < 0) continue;
#pragma unroll
        for (int r = 0; r < R; r++) buf[to[i] + r * Ns] = o[i][r];
    }
}

// all stages over the ng lines a workgroup has written to `buf` (not yet
// synchronised); the transforms are in `buf` afterwards, synchronised
__device__ __forceinline__ void fft_stages(double2* buf, int ng, const FFTAxis& A, int sign) {
    __syncthreads();
    int Ns = 1;
    for (int st = 0; st < A.nst; st++) {
        const int R = A.rad[st];
        if (R == 8) fft_stage<8>(buf, A, st, ng, Ns, sign);
        else if (R == 4) fft_stage<4>(buf, A, st, ng, Ns, sign);
        else if (R == 2) fft_stage<2>(buf, A, st, ng, Ns, sign);
        else if (R == 3) fft_stage<3>(buf, A, st, ng, Ns, sign);
        else fft_stage<5>(buf, A, st, ng, Ns, sign);
        __syncthreads();
        Ns *= R;
    }
}

// one workgroup: G lines of one axis, all stages in LDS; sign -1 forward, +1 inverse.
// Strided axes: a thread keeps one line (consecutive threads take consecutive
// lines, whose elements are adjacent in memory) and walks along it; along x the
// threads walk the line itself.
__global__ __launch_bounds__(256) void fft_lines(double2* __restrict__ data, FFTAxis A, int sign) {
    extern __shared__ double2 lds[];
    const int L = A.L, G = A.G;
    double2* const buf = lds;
    const int64_t l0 = (int64_t)blockIdx.x * G;
    const int ng = (int)min<int64_t>(G, A.nlines - l0);
    const int tid = threadIdx.x, nth = blockDim.x;
    if (A.S == 1) {
        for (int g = 0; g < ng; g++) {
            const int64_t l = l0 + g;
            const double2* line = data + (l % A.F) * A.sf + (l / A.F) * A.so;
            for (int j = tid; j < L; j += nth) buf[g * L + j] = line[j];
        }
    } else {
        const int g = tid % G, j0 = tid / G, js = nth / G;
        if (g < ng && j0 < js) {
            const int64_t l = l0 + g;
            const double2* line = data + (l % A.F) * A.sf + (l / A.F) * A.so;
            for (int j = j0; j < L; j += js) buf[g * L + j] = line[(int64_t)j * A.S];
        }
    }
    fft_stages(buf, ng, A, sign);
    if (A.S == 1) {
        for (int g = 0; g < ng; g++) {
            const int64_t l = l0 + g;
            double2* line = data + (l % A.F) * A.sf + (l / A.F) * A.so;
            for (int j = tid; j < L; j += nth) line[j] = buf[g * L + j];
        }
    } else {
        const int g = tid % G, j0 = tid / G, js = nth / G;
        if (g < ng && j0 < js) {
            const int64_t l = l0 + g;
            double2* line = data + (l % A.F) * A.sf + (l / A.F) * A.so;
            for (int j = j0; j < L; j += js) line[(int64_t)j * A.S] = buf[g * L + j];
        }
    }
}

// a node array as contiguous complex numbers
__global__ void to_complex(Grid G, const double* __restrict__ a, double2* __restrict__ c) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int x = (int)(i % G.nx);
    const int64_t row = i / G.nx;
    if (row < (int64_t)G.ny * G.nz) c[i] = make_double2(a[x + G.px * row], 0.0);
}

__global__ void real_part_scaled(int64_t n, const double2* __restrict__ c, double s, double* __restrict__ a) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) a[i] = c[i].x * s;
}

__device__ __forceinline__ int signed_k(int i, int n) { return i >= n / 2 + 1 ? i - n : i; }  // judge

__device__ __forceinline__ int shell_of(int x, int y, int z, int nx, int ny, int nz) {
    const int k1 = signed_k(x, nx), k2 = signed_k(y, ny), k3 = signed_k(z, nz);
    // |k|^2 <= 3 2^20 is exact in FP32, and below a square m^2 by at least 1, i.e. its
    // root is below m by more than half an ulp: the correctly rounded root truncates right
    return (int)sqrtf((float)(k1 * k1 + k2 * k2 + k3 * k3));
}

// x pass of a real field: G pairs of rows, row r at in + r in_pitch, into half
// spectra of nx/2 + 1 modes, row r at out + r out_pitch.  Rows 2p and 2p + 1 form
// one complex line Z = a + i b; with W = conj Z(-k), a_hat = (Z + W) / 2 and
// b_hat = -i (Z - W) / 2.  in may be out (in_pitch = 2 out_pitch): a workgroup
// reads its rows before it writes them.
__global__ __launch_bounds__(256) void rfft_rows(const double* in, int64_t in_pitch, int64_t nrows, FFTAxis A,
                                                 double2* out, int64_t out_pitch) {
    extern __shared__ double2 lds[];
    const int L = A.L, H = L / 2 + 1;
    const int64_t pairs = (nrows + 1) / 2, p0 = (int64_t)blockIdx.x * A.G;
    const int ng = (int)min<int64_t>(A.G, pairs - p0);
    for (int g = 0; g < ng; g++) {
        const int64_t r = 2 * (p0 + g);
        const bool two = r + 1 < nrows;
        for (int j = threadIdx.x; j < L; j += blockDim.x)
            lds[g * L + j] = make_double2(in[r * in_pitch + j], two ? in[(r + 1) * in_pitch + j] : 0.0);
    }
    fft_stages(lds, ng, A, -1);
    const double2* res = lds;
    for (int g = 0; g < ng; g++) {
        const int64_t r = 2 * (p0 + g);
        const bool two = r + 1 < nrows;
        for (int k = threadIdx.x; k < H; k += blockDim.x) {
            const double2 Z = res[g * L + k], V = res[g * L + (k == 0 ? 0 : L - k)];
            out[r * out_pitch + k] = make_double2(0.5 * (Z.x + V.x), 0.5 * (Z.y - V.y));
            if (two) out[(r + 1) * out_pitch + k] = make_double2(0.5 * (Z.y + V.y), 0.5 * (V.x - Z.x));
        }
    }
}

// what the z pass adds to the shell of a mode
enum { SHELL_ENERGY = 0,     // 0.5 |a|^2 on the half space k3 = 0..nz/2, weight 2 off k3 = 0 (the Nyquist plane
                             // included, as enesupe_cal counts it)
       SHELL_CROSS = 1,      // Re(a conj b) over all modes
       SHELL_CROSS_HALF = 2  // Re(a conj b) and the weights themselves on that half space (contribution,
                             // drop_analysis.f90:476-578); bins [sum | weight]
};
constexpr int SHELL_EL = FFT_POINTS / FFT_BLOCK;  // modes per thread of one workgroup's lines, at most

// z pass of the half spectra a (and b): G lines (kx, y) per round, transformed in
// LDS and added to the shells int|k| with the weight of the mode and its mirror
// image; workgroups take groups of lines in turn and leave one record of bins each
// (added to the one there if `more`), so that no bin is shared between workgroups.
template <int MODE>
__global__ __launch_bounds__(256) void zlines_shells(const double2* __restrict__ a, const double2* __restrict__ b,
                                                     FFTAxis A, int nx, int ny, int nz, double inv, int nshells,
                                                     int more, double* __restrict__ part) {
    extern __shared__ double2 lds[];
    const int L = A.L, G = A.G, tid = threadIdx.x, nbins = MODE == SHELL_CROSS_HALF ? 2 * nshells : nshells;
    double* bins = reinterpret_cast<double*>(lds + (size_t)G * L);
    double* rec = part + (int64_t)blockIdx.x * nbins;
    for (int s = tid; s < nbins; s += blockDim.x) bins[s] = more ? rec[s] : 0.0;
    const int64_t groups = (A.nlines + G - 1) / G;
    for (int64_t grp = blockIdx.x; grp < groups; grp += gridDim.x) {
        const int64_t l0 = grp * G;
        const int ng = (int)min<int64_t>(G, A.nlines - l0);
        auto transform = [&](const double2* __restrict__ src) {
            __syncthreads();  // the previous transform in LDS is read no more
            const int g = tid % G, j0 = tid / G, js = blockDim.x / G;
            if (g < ng && j0 < js) {
                const int64_t l = l0 + g;
                const double2* line = src + (l % A.F) * A.sf + (l / A.F) * A.so;
                for (int j = j0; j < L; j += js) lds[g * L + j] = line[(int64_t)j * A.S];
            }
            fft_stages(lds, ng, A, -1);
        };
        double2 va[SHELL_EL];
        const double2* res = lds;
        transform(a);
        if constexpr (MODE != SHELL_ENERGY) {
#pragma unroll
            for (int i = 0; i < SHELL_EL; i++) {
                const int m = tid + 256 * i;
                va[i] = m < ng * L ? res[m] : make_double2(0.0, 0.0);
            }
            transform(b);
        }
#pragma unroll
        for (int i = 0; i < SHELL_EL; i++) {
            const int m = tid + 256 * i;
            if (m >= ng * L) continue;
            const int g = (int)quotient(m, A.ml), z = m - g * L;
            const uint32_t l = (uint32_t)l0 + g;  // fewer than 2^22 lines
            const int y = (int)(l / (uint32_t)A.F), x = (int)(l - (uint32_t)y * A.F);
            const int s = shell_of(x, y, z, nx, ny, nz);
            if (s >= nshells) continue;
            const bool mirror = x != 0 && 2 * x != nx;  // -k is not among the stored modes
            double w;
            if constexpr (MODE == SHELL_CROSS) {
                w = mirror ? 2.0 : 1.0;
            } else {
                const int zm = z == 0 ? 0 : nz - z;
                w = (z <= nz / 2 ? (z == 0 ? 1.0 : 2.0) : 0.0) +
                    (mirror && zm <= nz / 2 ? (zm == 0 ? 1.0 : 2.0) : 0.0);
            }
            if (w == 0.0) continue;
            const double2 r = res[m];
            if constexpr (MODE == SHELL_ENERGY) {
                atomicAdd(&bins[s], 0.5 * ((r.x * r.x + r.y * r.y) * inv * inv) * w);
            } else {
                const double v = va[i].x * r.x + va[i].y * r.y;
                atomicAdd(&bins[s], MODE == SHELL_CROSS ? w * (v * inv * inv) : w * v);
                if constexpr (MODE == SHELL_CROSS_HALF) atomicAdd(&bins[nshells + s], w);
            }
        }
    }
    __syncthreads();
    for (int s = tid; s < nbins; s += blockDim.x) rec[s] = bins[s];
}

// out[s] = sum of the nrec workgroup records of bin s, fixed order, one workgroup per bin
__global__ __launch_bounds__(256) void shells_final(const double* __restrict__ part, int nrec, int nbins,
                                                    double* __restrict__ out) {
    __shared__ double sh[4];
    double v = 0.0;
    for (int r = threadIdx.x; r < nrec; r += 256) v += part[(int64_t)r * nbins + blockIdx.x];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = ((sh[0] + sh[1]) + sh[2]) + sh[3];
}

// keep the modes with lo <= int|k| < hi, zero the rest
__global__ void shell_mask(int nx, int ny, int nz, double2* __restrict__ a, int lo, int hi) {
    const int64_t n = (int64_t)nx * ny * nz;
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int x = (int)(i % nx), y = (int)((i / nx) % ny), z = (int)(i / ((int64_t)nx * ny));
    const int s = shell_of(x, y, z, nx, ny, nz);
    if (s < lo || s >= hi) a[i] = make_double2(0.0, 0.0);
}

// w_b = sum_a d_a (d_b phi d_a phi), b = 0..2, the stencil applied to the products
// at the neighbours (grad_tensor, drop_analysis.f90:1121-1217) of grad phi = sum c
// phi(x + c) / 10 (grad_cal); rows of w_b `pitch` apart, components `comp` apart.
// A workgroup stages phi over its tile + 2 nodes and forms grad phi over the tile + 1
// in LDS: two kernels gathering 14 neighbours through L2, with grad phi in memory
// between them, took 0.67 + 0.25 ms at 256^3, this one takes 0.34 ms.
constexpr int WTX = 32, WTY = 4, WTZ = 4, WNT = WTX * WTY * WTZ;
template <int Q0, int Q1, typename Fn> __device__ __forceinline__ void sford(Fn&& fn) {
    if constexpr (Q0 < Q1) {
        fn(std::integral_constant<int, Q0>{});
        sford<Q0 + 1, Q1>(fn);
    }
}
__global__ __launch_bounds__(WNT) void div_korteweg(Grid G, const double* __restrict__ phi,
                                                    double* __restrict__ w, int64_t pitch, int64_t comp, int tiles_x,
                                                    int tiles_y) {
    constexpr int HX2 = WTX + 4, HY2 = WTY + 4, HZ2 = WTZ + 4, H2 = HX2 * HY2 * HZ2;
    constexpr int HX1 = WTX + 2, HY1 = WTY + 2, HZ1 = WTZ + 2, H1 = HX1 * HY1 * HZ1;
    __shared__ double sp[H2];
    __shared__ double sg[3][H1];
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % tiles_x) * WTX, y0 = ((tile / tiles_x) % tiles_y) * WTY,
              z0 = (tile / (tiles_x * tiles_y)) * WTZ;
    const bool small = nx <= WTX || ny <= WTY || nz <= WTZ;  // a tile's halo may wrap more than once
    auto wrap = [small](int v, int n) {
        if (small) {
            v %= n;
            return v < 0 ? v + n : v;
        }
        return v < 0 ? v + n : (v >= n ? v - n : v);
    };
    for (int h = threadIdx.x; h < H2; h += WNT) {
        const int gx = wrap(x0 - 2 + h % HX2, nx), gy = wrap(y0 - 2 + (h / HX2) % HY2, ny),
                  gz = wrap(z0 - 2 + h / (HX2 * HY2), nz);
        sp[h] = phi[G.node(gx, gy, gz)];
    }
    __syncthreads();
    for (int h = threadIdx.x; h < H1; h += WNT) {
        const int c = h % HX1 + HX2 * ((h / HX1) % HY1 + HY2 * (h / (HX1 * HY1)));
        double g0 = 0.0, g1 = 0.0, g2 = 0.0;
        sford<1, 15>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            using D = Dir<q>;
            const double v = sp[c + (1 + D::cx) + HX2 * ((1 + D::cy) + HY2 * (1 + D::cz))];
            g0 = acc<D::cx>(g0, v);
            g1 = acc<D::cy>(g1, v);
            g2 = acc<D::cz>(g2, v);
        });
        sg[0][h] = div_const(g0, 10.0, 0.1);
        sg[1][h] = div_const(g1, 10.0, 0.1);
        sg[2][h] = div_const(g2, 10.0, 0.1);
    }
    __syncthreads();
    const int tx = threadIdx.x % WTX, ty = (threadIdx.x / WTX) % WTY, tz = threadIdx.x / (WTX * WTY);
    const int x = x0 + tx, y = y0 + ty, z = z0 + tz;
    if (x >= nx || y >= ny || z >= nz) return;
    double d0 = 0.0, d1 = 0.0, d2 = 0.0;
    sford<1, 15>([&](auto qc) {
        constexpr int q = decltype(qc)::value;
        using D = Dir<q>;
        const int h = (tx + 1 + D::cx) + HX1 * ((ty + 1 + D::cy) + HY1 * (tz + 1 + D::cz));
        const double g0 = sg[0][h], g1 = sg[1][h], g2 = sg[2][h], cg = cdot<q>(g0, g1, g2);
        d0 += g0 * cg;
        d1 += g1 * cg;
        d2 += g2 * cg;
    });
    double* const o = w + x + pitch * (y + (int64_t)ny * z);
    o[0] = div_const(d0, 10.0, 0.1);
    o[comp] = div_const(d1, 10.0, 0.1);
    o[2 * comp] = div_const(d2, 10.0, 0.1);
}

// ------------------------------------------------------------------ host side

struct FFTPlan {
    int n[3] = {0, 0, 0};
    FFTAxis ax[3];
    double2* tw = nullptr;  // the three twiddle tables, back to back
    ~FFTPlan() {
        if (tw) (void)hipFree(tw);
    }
};

int factor(int L, int* rad, int* nst) {
    *nst = 0;
    int m = L;
    for (const int R : {8, 4, 2, 3, 5}) {
        while (m % R == 0 && !(R == 8 && m % 32 == 16)) {  // 16 = 4 x 4, not 8 x 2
            if (*nst >= FFT_MAX_STAGES) return -1;
            rad[(*nst)++] = R;
            m /= R;
        }
    }
    return m == 1 ? 0 : -1;
}

int make_plan(int nx, int ny, int nz, FFTPlan& P) {
    const int ns[3] = {nx, ny, nz};
    for (int a = 0; a < 3; a++) {
        if (ns[a] > FFT_MAX_LINE || factor(ns[a], P.ax[a].rad, &P.ax[a].nst))
            return drp_fail(DRP_ERR_UNSUPPORTED, "FFT diagnostics need extents that are products of 2, 3 and 5, "
                                                 "at most %d (got %d)", FFT_MAX_LINE, ns[a]);
        P.n[a] = ns[a];
    }
    HIP_TRYS(hipMalloc((void**)&P.tw, (size_t)(nx + ny + nz) * sizeof(double2)));
    std::vector<double2> t;
    for (int a = 0; a < 3; a++)
        for (int j = 0; j < ns[a]; j++) {
            const long double th = -2.0L * 3.14159265358979323846264338327950288L * (long double)j / (long double)ns[a];
            t.push_back(make_double2((double)cosl(th), (double)sinl(th)));
        }
    HIP_TRYS(hipMemcpy(P.tw, t.data(), t.size() * sizeof(double2), hipMemcpyHostToDevice));
    const int64_t nxy = (int64_t)nx * ny;
    // x: lines contiguous; y: lines (x, z), stride nx; z: lines (x, y), stride nx ny
    P.ax[0].L = nx; P.ax[0].S = 1;   P.ax[0].nlines = nxy / nx * nz; P.ax[0].F = 1; P.ax[0].sf = 0; P.ax[0].so = nx;
    P.ax[1].L = ny; P.ax[1].S = nx;  P.ax[1].nlines = (int64_t)nx * nz; P.ax[1].F = nx; P.ax[1].sf = 1; P.ax[1].so = nxy;
    P.ax[2].L = nz; P.ax[2].S = nxy; P.ax[2].nlines = nxy; P.ax[2].F = nx; P.ax[2].sf = 1; P.ax[2].so = nx;
    P.ax[0].tw = P.tw;
    P.ax[1].tw = P.tw + nx;
    P.ax[2].tw = P.tw + nx + ny;
    auto magic = [](int d) { return d == 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + d - 1) / d); };
    for (int a = 0; a < 3; a++) {
        FFTAxis& A = P.ax[a];
        A.G = std::max(1, std::min(16, FFT_POINTS / A.L));
        A.ml = magic(A.L);
        for (int st = 0, Ns = 1; st < A.nst; Ns *= A.rad[st++]) {
            A.mm[st] = magic(A.L / A.rad[st]);
            A.mn[st] = magic(Ns);
        }
    }
    return DRP_OK;
}

hipError_t fft3d(const FFTPlan& P, double2* data, int sign, hipStream_t st) {
    for (int a = 0; a < 3; a++) {
        const FFTAxis& A = P.ax[a];
        const int64_t blocks = (A.nlines + A.G - 1) / A.G;
        const size_t lds = (size_t)A.G * A.L * sizeof(double2);
        hipLaunchKernelGGL(fft_lines, dim3((unsigned)blocks), dim3(256), lds, st, data, A, sign);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// device buffer released on scope exit
struct DevMem {
    void* p = nullptr;
    ~DevMem() {
        if (p) (void)hipFree(p);
    }
};

int velocity_view(drp_lattice* L, const double** mac) {
    if (L->cfg.precision == DRP_FP64) {
        *mac = (const double*)L->mac[L->cur];
        return DRP_OK;
    }
    return fp32_macro_fp64_view(L, mac);
}

// forward transforms of u1, u2, u3 into c[3][n] (unnormalised)
int transform_velocity(drp_lattice* L, const FFTPlan& P, double2* c) {
    const double* mac = nullptr;
    int rc = velocity_view(L, &mac);
    if (rc) return rc;
    const int64_t n = L->n;
    const unsigned nb = (unsigned)((n + 255) / 256);
    for (int k = 0; k < 3; k++) {
        hipLaunchKernelGGL(to_complex, dim3(nb), dim3(256), 0, L->stream, L->G, mac + (2 + k) * L->G.ns, c + k * n);
        HIP_TRYS(hipGetLastError());
        HIP_TRYS(fft3d(P, c + k * n, -1, L->stream));
    }
    return DRP_OK;
}

}  // namespace

// The spectra's plan, twiddles and work space of one lattice, kept from its first
// spectrum until it is destroyed: one half spectrum (8.5 B per node) for the energy
// spectrum, two for the cross spectrum, four for the interaction (34 B per node, 5 %
// of an FP64 lattice's own memory), and the shell records.  Allocating and freeing the
// work space per call (48 to 120 B per node of full complex transforms) took most of a
// call: 10 ms for the analysis of a 256^3 state with an idle memory pool, up to 190 ms
// when the freed blocks were still in use elsewhere.
struct drp_diag {
    FFTPlan P;
    FFTAxis y, z;          // half-spectrum lines
    int64_t pitch = 0;     // complex numbers per row: nx/2 + 1 rounded up to 128 bytes
    int64_t rows = 0;      // ny nz
    double2* half = nullptr;    // `spectra` half spectra
    int spectra = 0;
    double* part = nullptr;     // workgroup records, then the summed bins
    size_t part_cap = 0;
    ~drp_diag() {
        if (half) (void)hipFree(half);
        if (part) (void)hipFree(part);
    }
    double2* spectrum(int k) { return half + k * rows * pitch; }
};

void diag_free(drp_lattice* L) {
    delete L->diag;
    L->diag = nullptr;
}

namespace {

// Workgroups of the z pass.  The lines and the bins of one take 33 KiB of LDS at 256^3, so
// four fit a CU: of 1280 the last 256 start when others end.  1024 are no better: energy
// spectrum 807 us with 1280, 834 with 1024, interaction 2081 and 2044 (768: 771 and 2154;
// 128^3 212 and 209, 415 and 416).
constexpr int SHELL_WGS = 1280;

// L->diag with room for `spectra` half spectra
int diag_get(drp_lattice* L, int spectra, drp_diag** out) {
    if (!L->diag) {
        drp_diag* D = new (std::nothrow) drp_diag();
        if (!D) return drp_fail(DRP_ERR_ALLOC, "host allocation failed");
        const drp_config& c = L->cfg;
        int rc = make_plan(c.nx, c.ny, c.nz, D->P);
        if (!rc) {
            const int hx = c.nx / 2 + 1;
            D->pitch = (hx + 7) / 8 * 8;
            D->rows = (int64_t)c.ny * c.nz;
            D->y = D->P.ax[1];
            D->y.S = D->pitch;
            D->y.nlines = (int64_t)hx * c.nz;
            D->y.F = hx;
            D->y.so = D->pitch * c.ny;
            D->z = D->P.ax[2];
            D->z.S = D->pitch * c.ny;
            D->z.nlines = (int64_t)hx * c.ny;
            D->z.F = hx;
            D->z.so = D->pitch;
        }
        if (rc) {
            delete D;
            return rc;
        }
        L->diag = D;
    }
    drp_diag* D = L->diag;
    if (D->spectra < spectra) {
        if (D->half) (void)hipFree(D->half);
        D->half = nullptr;
        D->spectra = 0;
        HIP_TRYS(hipMalloc((void**)&D->half, spectra * (size_t)(D->rows * D->pitch) * sizeof(double2)));
        D->spectra = spectra;
    }
    *out = L->diag;
    return DRP_OK;
}

// x and y passes of a real field with row pitch in_pitch into half spectrum k
int half_transform(drp_diag* D, const double* in, int64_t in_pitch, int k, hipStream_t st) {
    const FFTAxis& X = D->P.ax[0];
    double2* out = D->spectrum(k);
    const int64_t pairs = (D->rows + 1) / 2;
    hipLaunchKernelGGL(rfft_rows, dim3((unsigned)((pairs + X.G - 1) / X.G)), dim3(256),
                       (size_t)X.G * X.L * sizeof(double2), st, in, in_pitch, D->rows, X, out, D->pitch);
    HIP_TRYS(hipGetLastError());
    const FFTAxis& Y = D->y;
    hipLaunchKernelGGL(fft_lines, dim3((unsigned)((Y.nlines + Y.G - 1) / Y.G)), dim3(256),
                       (size_t)Y.G * Y.L * sizeof(double2), st, out, Y, -1);
    HIP_TRYS(hipGetLastError());
    return DRP_OK;
}

// the records of the z pass: their number for nbins bins, room for them and the sums
int shell_records(drp_diag* D, int nbins, int* wgs) {
    const int64_t groups = (D->z.nlines + D->z.G - 1) / D->z.G;
    // a few thousand bins per workgroup would outgrow the transforms: fewer workgroups then
    *wgs = (int)std::min<int64_t>(groups, std::max<int64_t>(256, std::min<int64_t>(SHELL_WGS, (int64_t)SHELL_WGS * 512 / nbins)));
    const size_t need = ((size_t)*wgs + 1) * nbins;
    if (D->part_cap < need) {
        if (D->part) (void)hipFree(D->part);
        D->part = nullptr;
        D->part_cap = 0;
        HIP_TRYS(hipMalloc((void**)&D->part, need * sizeof(double)));
        D->part_cap = need;
    }
    return DRP_OK;
}

// z pass of half spectrum 0 (and `other`), added to the records
template <int MODE>
int shell_pass(drp_lattice* L, drp_diag* D, int other, double inv, int nshells, int nbins, int wgs, bool more) {
    const FFTAxis& Z = D->z;
    const size_t lds = (size_t)Z.G * Z.L * sizeof(double2) + nbins * sizeof(double);
    // (thousands of shells need up to 96 KiB of the CU's 160)
    if (lds > 64 * 1024)
        HIP_TRYS(hipFuncSetAttribute(reinterpret_cast<const void*>(&zlines_shells<MODE>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((zlines_shells<MODE>), dim3(wgs), dim3(256), lds, L->stream, D->spectrum(0), D->spectrum(other), Z,
                       L->cfg.nx, L->cfg.ny, L->cfg.nz, inv, nshells, more ? 1 : 0, D->part);
    HIP_TRYS(hipGetLastError());
    return DRP_OK;
}

// the summed bins to the host
int shell_sums(drp_lattice* L, drp_diag* D, int nbins, int wgs, double* host) {
    double* out = D->part + (size_t)wgs * nbins;
    hipLaunchKernelGGL(shells_final, dim3(nbins), dim3(256), 0, L->stream, D->part, wgs, nbins, out);
    HIP_TRYS(hipGetLastError());
    HIP_TRYS(hipMemcpyAsync(host, out, (size_t)nbins * sizeof(double), hipMemcpyDeviceToHost, L->stream));
    HIP_TRYS(hipStreamSynchronize(L->stream));
    return DRP_OK;
}

// w_b, b = 0..2, into the half spectra 1..3, in rows of 2 pitch doubles
int korteweg_divergence(drp_lattice* L, drp_diag* D, const double* phi) {
    const Grid& G = L->G;
    const int tx = (G.nx + WTX - 1) / WTX, ty = (G.ny + WTY - 1) / WTY, tz = (G.nz + WTZ - 1) / WTZ;
    hipLaunchKernelGGL(div_korteweg, dim3((unsigned)(tx * ty * tz)), dim3(WNT), 0, L->stream, G, phi,
                       (double*)D->spectrum(1), 2 * D->pitch, 2 * D->pitch * D->rows, tx, ty);
    HIP_TRYS(hipGetLastError());
    return DRP_OK;
}

}  // namespace

// FFT round trip on a caller's complex field (for tests of the transform itself):
// data[n] complex as interleaved (re, im), sign -1 forward, +1 inverse (unnormalised).
extern "C" int drp_fft3d(int nx, int ny, int nz, double* data, int sign) {
    if (!data || nx < 1 || ny < 1 || nz < 1 || (sign != -1 && sign != 1)) return drp_fail(DRP_ERR_ARG, "bad FFT arguments");
    FFTPlan P;
    int rc = make_plan(nx, ny, nz, P);
    if (rc) return rc;
    const int64_t n = (int64_t)nx * ny * nz;
    DevMem d;
    HIP_TRYS(hipMalloc(&d.p, (size_t)n * sizeof(double2)));
    HIP_TRYS(hipMemcpy(d.p, data, (size_t)n * sizeof(double2), hipMemcpyHostToDevice));
    HIP_TRYS(fft3d(P, (double2*)d.p, sign, nullptr));
    HIP_TRYS(hipMemcpy(data, d.p, (size_t)n * sizeof(double2), hipMemcpyDeviceToHost));
    return DRP_OK;
}

constexpr int MAX_SHELLS = 8192;  // shell bins of one workgroup in LDS

extern "C" int drp_energy_spectrum(drp_lattice* L, double* E, int nshells) {
    if (!L || !E || nshells < 1 || nshells > MAX_SHELLS) return drp_fail(DRP_ERR_ARG, "bad spectrum arguments");
    if (!L->initialized) return drp_fail(DRP_ERR_STATE, "lattice not initialised");
    drp_diag* D = nullptr;
    int rc = diag_get(L, 1, &D);
    if (rc) return rc;
    const double* mac = nullptr;
    int wgs = 0;
    rc = velocity_view(L, &mac);
    if (!rc) rc = shell_records(D, nshells, &wgs);
    for (int k = 0; k < 3 && !rc; k++) {
        rc = half_transform(D, mac + (2 + k) * L->G.ns, L->G.px, 0, L->stream);
        if (!rc) rc = shell_pass<SHELL_ENERGY>(L, D, 0, 1.0 / (double)L->n, nshells, nshells, wgs, k > 0);
    }
    return rc ? rc : shell_sums(L, D, nshells, wgs, E);
}

extern "C" int drp_filter_velocity(drp_lattice* L, int kind, int k, double* u1, double* u2, double* u3, size_t n_) {
    if (!L || !u1 || !u2 || !u3) return drp_fail(DRP_ERR_ARG, "null argument");
    if (kind != DRP_FILTER_LOW_PASS && kind != DRP_FILTER_SHELL) return drp_fail(DRP_ERR_ARG, "unknown filter %d", kind);
    if (n_ != (size_t)L->n) return drp_fail(DRP_ERR_ARG, "size %zu != %lld nodes", n_, (long long)L->n);
    if (!L->initialized) return drp_fail(DRP_ERR_STATE, "lattice not initialised");
    const drp_config& c = L->cfg;
    FFTPlan P;
    int rc = make_plan(c.nx, c.ny, c.nz, P);
    if (rc) return rc;
    const int64_t n = L->n;
    DevMem cu, out;
    HIP_TRYS(hipMalloc(&cu.p, 3 * (size_t)n * sizeof(double2)));
    HIP_TRYS(hipMalloc(&out.p, (size_t)n * sizeof(double)));
    rc = transform_velocity(L, P, (double2*)cu.p);
    if (rc) return rc;
    // low_pass keeps int|k| + 1 <= k_low, i.e. int|k| < k; the band-pass keeps int|k| == k
    const int lo = kind == DRP_FILTER_LOW_PASS ? 0 : k, hi = kind == DRP_FILTER_LOW_PASS ? k : k + 1;
    const unsigned nb = (unsigned)((n + 255) / 256);
    double* dst[3] = {u1, u2, u3};
    for (int a = 0; a < 3; a++) {
        double2* ca = (double2*)cu.p + a * n;
        hipLaunchKernelGGL(shell_mask, dim3(nb), dim3(256), 0, L->stream, c.nx, c.ny, c.nz, ca, lo, hi);
        HIP_TRYS(hipGetLastError());
        HIP_TRYS(fft3d(P, ca, +1, L->stream));
        hipLaunchKernelGGL(real_part_scaled, dim3(nb), dim3(256), 0, L->stream, n, (const double2*)ca, 1.0 / (double)n,
                           (double*)out.p);
        HIP_TRYS(hipGetLastError());
        rc = dense_to_host(L, (const double*)out.p, dst[a]);
        if (rc) return rc;
    }
    return DRP_OK;
}

extern "C" int drp_scale_interaction(drp_lattice* L, double* C, int nshells) {
    if (!L || !C || nshells < 1 || nshells > MAX_SHELLS) return drp_fail(DRP_ERR_ARG, "bad interaction arguments");
    if (!L->initialized) return drp_fail(DRP_ERR_STATE, "lattice not initialised");
    drp_diag* D = nullptr;
    int rc = diag_get(L, 4, &D);
    if (rc) return rc;
    const double* mac = nullptr;
    int wgs = 0;
    rc = velocity_view(L, &mac);
    if (!rc) rc = shell_records(D, nshells, &wgs);
    if (!rc) rc = korteweg_divergence(L, D, mac);
    for (int b = 0; b < 3 && !rc; b++) {
        rc = half_transform(D, (const double*)D->spectrum(1 + b), 2 * D->pitch, 1 + b, L->stream);
        if (!rc) rc = half_transform(D, mac + (2 + b) * L->G.ns, L->G.px, 0, L->stream);
        if (!rc) rc = shell_pass<SHELL_CROSS>(L, D, 1 + b, 1.0 / (double)L->n, nshells, nshells, wgs, b > 0);
    }
    std::vector<double> h(nshells);
    if (!rc) rc = shell_sums(L, D, nshells, wgs, h.data());
    if (rc) return rc;
    for (int s = 0; s < nshells; s++) C[s] = L->cfg.kappa_g * h[s];
    return DRP_OK;
}

extern "C" int drp_phi_contribution(drp_lattice* L, double* C, int nshells, double* bands) {
    if (!L || !C || !bands) return drp_fail(DRP_ERR_ARG, "null argument");
    if (!L->initialized) return drp_fail(DRP_ERR_STATE, "lattice not initialised");
    const drp_config& c = L->cfg;
    const int nb = c.nx / 2 + 1;  // the reference's (xmax+1)/2 + 1 shells
    if (nshells < 1 || nshells > nb) return drp_fail(DRP_ERR_ARG, "nshells %d not in 1..%d", nshells, nb);
    drp_diag* D = nullptr;
    int rc = diag_get(L, 2, &D);
    if (rc) return rc;
    const double* mac = nullptr;
    int wgs = 0;
    rc = velocity_view(L, &mac);
    if (!rc) rc = shell_records(D, 2 * nb, &wgs);
    const int kinds[2] = {DRP_DERIVED_ADVECTION, DRP_DERIVED_CHEMICAL_POTENTIAL};
    for (int k = 0; k < 2 && !rc; k++) {
        double* field = (double*)D->spectrum(k);
        HIP_TRYS(launch_derived_fp64(L->G, L->phys, mac, kinds[k], field, 2 * D->pitch, L->stream));
        rc = half_transform(D, field, 2 * D->pitch, k, L->stream);
    }
    if (!rc) rc = shell_pass<SHELL_CROSS_HALF>(L, D, 1, 1.0, nb, 2 * nb, wgs, false);
    std::vector<double> h(2 * (size_t)nb);
    if (!rc) rc = shell_sums(L, D, 2 * nb, wgs, h.data());
    if (rc) return rc;
    std::vector<double> res(nb);
    for (int s = 0; s < nb; s++) res[s] = h[nb + s] > 0.0 ? h[s] / h[nb + s] : 0.0;
    for (int s = 0; s < nshells; s++) C[s] = res[s];
    // energy_large: i = 2..4, energy_medium: i = 5..10, energy_small: i = 11 .. nb (1-based)
    double all = 0.0, large = 0.0, medium = 0.0, small = 0.0;
    for (int s = 1; s <= 3 && s < nb; s++) {
        large = large + res[s];
        all = all + res[s];
    }
    for (int s = 4; s <= 9 && s < nb; s++) {
        medium = medium + res[s];
        all = all + res[s];
    }
    for (int s = 10; s < nb; s++) {
        small = small + res[s];
        all = all + res[s];
    }
    bands[0] = all * (-1.0);
    bands[1] = large * (-1.0);
    bands[2] = medium * (-1.0);
    bands[3] = small * (-1.0);
    return DRP_OK;
}
