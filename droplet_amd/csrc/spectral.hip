// spectral.hip — linear forcing of the low Fourier shells for forced isotropic
// turbulence (program/lbm_drop_iht_xy.f90:722-841, externalforce).
//
// The reference transforms u with a full 3-D r2c FFT (2decomp + FFTW), keeps the
// modes with 1 <= |k| < kc (integer mode numbers, kc = 3), computes their energy
//   E_low = 1/2 sum_{k in S} |u_hat_k|^2,   u_hat = FFT(u) / N^3,
// and transforms F_hat_k = (eps / (2 E_low)) u_hat_k (zero off S) back, so that
// the injected power <F . u> is eps by construction.
//
// Only the few modes of S (|k_a| <= K = kc - 1 per axis) enter, so here the
// transform is a truncated, separable DFT instead of three full FFTs:
//   rows_fwd  A(kx, y, z)   = sum_x u e^{-2 pi i kx x/nx}        kx = 0..K (u real:
//                                                               -kx is conj(kx))
//   cols_fwd  B(kx, ky, z)  = sum_y A e^{-2 pi i ky y/ny}        ky = -K..K
//   zsum      u_hat(k)      = sum_z B e^{-2 pi i kz z/nz} / N^3
//   force     E_low and the coefficients C(k) = eps / (2 E_low) u_hat(k) on S,
//             G(kx, ky)     = sum_kz C e^{+2 pi i kz z/nz}       for its plane z,
//             H(kx, y)      = sum_ky G e^{+2 pi i ky y/ny}       for its rows,
//             F(x, y, z)    = Re H(0) + 2 sum_{kx>0} Re(H(kx) e^{+2 pi i kx x/nx})
// The first and last passes touch every node once (read u, write F); the others
// work on N^2 rows or less, one wavefront per output with the lanes over the
// summed axis.  The coefficients are few (225 for kc = 3), so every workgroup of the
// last pass forms what it needs of C, G and H by itself: as passes of their own these
// took three launches and 19 us a step at 192^3 and below.  E_low = 0 gives F = 0 (the
// reference would divide by zero).
//
// The same passes with unit coefficients on the shells klo <= int|k| < khi give
// the band-pass of u that advects phi in the scale-separated model
// (program/lbm_drop_scale_xy.f90:846-903, low_pass; u_hat = FFT(u)/N^3 there too).
#include "kernels.h"

namespace drp {

namespace {

constexpr int SF_BLOCK = 256;

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// e^{s 2 pi i m / n} from the table tw[j] = (cos 2 pi j/n, sin 2 pi j/n), s = +-1.
// Every caller has |m| <= K (n - 1) with K <= 4, so m is reduced into [0, n) by a
// few compares instead of a (64-bit) integer remainder.
__device__ __forceinline__ double2 twiddle(const double2* tw, int m, int n, int s) {
    int j = m;
    while (j >= n) j -= n;
    while (j < 0) j += n;
    const double2 t = tw[j];
    return make_double2(t.x, s * t.y);
}

// Sum of NV per-lane values over the 64 lanes of a wavefront with about 2 SL shuffles
// (SL = NV rounded up to 16 or 32) instead of 6 NV: at each offset 32, 16, .. a lane
// keeps one half of its values (the upper one when lane & offset) and adds the
// partner's copy of that half; when one value is left, lane l holds value
// l / (64 / SL), and the remaining offsets complete it.
template <int O, int HALF, int SL> __device__ __forceinline__ void halve(double (&v)[SL], int lane) {
    const bool up = (lane & O) != 0;
#pragma unroll
    for (int i = 0; i < HALF; i++) {
        const double keep = up ? v[i + HALF] : v[i];
        const double give = up ? v[i] : v[i + HALF];
        v[i] = keep + __shfl_xor(give, O, 64);
    }
    if constexpr (HALF > 1) halve<O / 2, HALF / 2>(v, lane);
}

template <int SL> __device__ __forceinline__ double wave_sums(double (&v)[SL], int lane) {
    static_assert(SL == 16 || SL == 32, "16 or 32 values");
    halve<32, SL / 2>(v, lane);
#pragma unroll
    for (int o = 32 / SL; o > 0; o /= 2) v[0] += __shfl_xor(v[0], o, 64);
    return v[0];
}

// pass 1: a wavefront takes RF_ROWS (y, z) rows in turn; the loads of CH x-iterations
// are issued together before their products are accumulated, and rows of up to 64 CH
// nodes keep their twiddles in registers.  Measured at 256^3, FP64 / FP32: one row per
// wavefront with kx = 0 multiplied like the others 97 / 131 us (128^3 FP32: 28), this 85 us (128^3 FP32: 19); with the
// next row's loads in flight during the sums 121 us (fewer wavefronts fit).
constexpr int RF_ROWS = 4;
template <int K, typename T>
__global__ __launch_bounds__(SF_BLOCK) void sf_rows_fwd(int nx, int px, int ny, int nz, const T* __restrict__ u1,
                                                        const T* __restrict__ u2, const T* __restrict__ u3,
                                                        const double2* __restrict__ twx, double2* __restrict__ A) {
    constexpr int PC = 2 * K + 1, NV = 3 * PC, SL = NV <= 16 ? 16 : 32, CH = 4;  // per component: re 0, (re, im) 1..K
    const int lane = threadIdx.x & 63;
    const long rows = (long)ny * nz;
    const long row0 = ((long)blockIdx.x * (SF_BLOCK / 64) + (threadIdx.x >> 6)) * RF_ROWS;
    const T* u[3] = {u1, u2, u3};
    double2 e[CH][K];
    auto twiddles = [&](int x0) {
#pragma unroll
        for (int j = 0; j < CH; j++) {
            const int x = x0 + 64 * j + lane;
#pragma unroll
            for (int k = 1; k <= K; k++) e[j][k - 1] = twiddle(twx, k * (x < nx ? x : 0), nx, -1);
        }
    };
    twiddles(0);
    for (long row = row0; row < min(row0 + RF_ROWS, rows); row++) {  // uniform per wavefront
        double acc[SL];
#pragma unroll
        for (int i = 0; i < SL; i++) acc[i] = 0.0;
        for (int x0 = 0; x0 < nx; x0 += 64 * CH) {
            if (nx > 64 * CH) twiddles(x0);
            double v[CH][3];
#pragma unroll
            for (int j = 0; j < CH; j++) {
                const int x = x0 + 64 * j + lane;
                const bool ok = x < nx;
                const long s = row * px + (ok ? x : 0);
#pragma unroll
                for (int c = 0; c < 3; c++) v[j][c] = ok ? (double)u[c][s] : 0.0;
            }
#pragma unroll
            for (int j = 0; j < CH; j++)
#pragma unroll
                for (int c = 0; c < 3; c++) {
                    acc[c * PC] += v[j][c];
#pragma unroll
                    for (int k = 1; k <= K; k++) {
                        acc[c * PC + 2 * k - 1] += v[j][c] * e[j][k - 1].x;
                        acc[c * PC + 2 * k] += v[j][c] * e[j][k - 1].y;
                    }
                }
        }
        const double t = wave_sums<SL>(acc, lane);
        const int idx = lane / (64 / SL);
        if (lane % (64 / SL) == 0 && idx < NV) {
            const int c = idx / PC, i = idx - c * PC;  // i = 0: re of kx = 0, whose im is 0
            double* out = reinterpret_cast<double*>(A + (row * 3 + c) * (K + 1));
            out[i == 0 ? 0 : i + 1] = t;
            if (i == 0) out[1] = 0.0;
        }
    }
}

// pass 2: one wavefront per (z, c, kx, ky), lanes over y
template <int K>
__global__ __launch_bounds__(SF_BLOCK) void sf_cols_fwd(int ny, int nz, const double2* __restrict__ A,
                                                        const double2* __restrict__ twy, double2* __restrict__ B) {
    constexpr int NK = 2 * K + 1, NB = 3 * (K + 1) * NK;
    const int lane = threadIdx.x & 63;
    const long w = (long)blockIdx.x * (SF_BLOCK / 64) + (threadIdx.x >> 6);
    if (w >= (long)nz * NB) return;  // uniform per wavefront
    const int b = (int)(w % NB), z = (int)(w / NB);
    const int ky = b % NK - K, kx = (b / NK) % (K + 1), c = b / (NK * (K + 1));
    double sr = 0.0, si = 0.0;
    for (int y = lane; y < ny; y += 64) {
        const double2 p = cmul(A[(((long)z * ny + y) * 3 + c) * (K + 1) + kx], twiddle(twy, ky * y, ny, -1));
        sr += p.x;
        si += p.y;
    }
    for (int off = 32; off > 0; off >>= 1) {
        sr += __shfl_xor(sr, off, 64);
        si += __shfl_xor(si, off, 64);
    }
    if (lane == 0) B[w] = make_double2(sr, si);  // [z][c][kx][ky]
}

// pass 3a: one wavefront per mode (c, kx, ky, kz), lanes over z: u_hat into U
template <int K>
__global__ __launch_bounds__(SF_BLOCK) void sf_zsum(int nx, int ny, int nz, const double2* __restrict__ B,
                                                    const double2* __restrict__ twz, double2* __restrict__ U) {
    constexpr int NK = 2 * K + 1, NB = 3 * (K + 1) * NK, NC = NB * NK;
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * (SF_BLOCK / 64) + (threadIdx.x >> 6);
    if (t >= NC) return;  // uniform per wavefront
    const int kz = t % NK - K, b = t / NK;
    double sr = 0.0, si = 0.0;
    for (int z = lane; z < nz; z += 64) {
        const double2 p = cmul(B[(long)z * NB + b], twiddle(twz, kz * z, nz, -1));
        sr += p.x;
        si += p.y;
    }
    for (int off = 32; off > 0; off >>= 1) {
        sr += __shfl_xor(sr, off, 64);
        si += __shfl_xor(si, off, 64);
    }
    const double inv = 1.0 / ((double)nx * ny * nz);
    if (lane == 0) U[t] = make_double2(sr * inv, si * inv);
}

// pass 4: SF_ROWS rows of one z plane per workgroup.  The coefficients of the kept
// modes k2lo <= |k|^2 < k2hi, the others zeroed: forcing (band = 0) scaled by eps /
// (2 E_low) with E_low the energy of the kept modes, band-pass (band = 1) unscaled;
// then the inverse transform along z for the plane, along y for the rows, and along
// x with the lanes over x and the rows of a wavefront sharing the twiddles.
constexpr int SF_ROWS = 16;
template <int K>
__global__ __launch_bounds__(SF_BLOCK) void sf_force(int nx, int px, int ny, int nz, int k2lo, int k2hi, int band,
                                                     double eps, const double2* __restrict__ U,
                                                     const double2* __restrict__ twx, const double2* __restrict__ twy,
                                                     const double2* __restrict__ twz, double* __restrict__ elow_out,
                                                     double* __restrict__ fx, double* __restrict__ fy,
                                                     double* __restrict__ fz) {
    constexpr int NK = 2 * K + 1, NH = 3 * (K + 1), NB = NH * NK, NC = NB * NK, W = SF_BLOCK / 64;
    __shared__ double2 s_u[NC], s_g[NB], s_h[SF_ROWS][NH];
    __shared__ double s_e[W];
    const int chunks = (ny + SF_ROWS - 1) / SF_ROWS;
    const int z = blockIdx.x / chunks, y0 = (blockIdx.x - z * chunks) * SF_ROWS, nr = min(SF_ROWS, ny - y0);
    auto k_squared = [](int t) {
        const int kz = t % NK - K, b = t / NK;
        const int ky = b % NK - K, kx = (b / NK) % (K + 1);
        return kx * kx + ky * ky + kz * kz;
    };
    double e = 0.0;
    for (int t = threadIdx.x; t < NC; t += SF_BLOCK) {
        const double2 s = U[t];
        const int k2 = k_squared(t);
        const bool in = k2 >= k2lo && k2 < k2hi;
        s_u[t] = in ? s : make_double2(0.0, 0.0);
        if (in) e += ((t / NK / NK) % (K + 1) == 0 ? 0.5 : 1.0) * (s.x * s.x + s.y * s.y);
    }
    for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off, 64);
    if ((threadIdx.x & 63) == 0) s_e[threadIdx.x >> 6] = e;
    __syncthreads();
    double elow = 0.0;
    for (int w = 0; w < W; w++) elow += s_e[w];
    const double alpha = band ? 1.0 : (elow > 0.0 ? 0.5 * eps / elow : 0.0);
    if (blockIdx.x == 0 && threadIdx.x == 0) *elow_out = elow;
    for (int t = threadIdx.x; t < NB; t += SF_BLOCK) {  // [c][kx][ky]
        double2 s = make_double2(0.0, 0.0);
        for (int kz = -K; kz <= K; kz++) {
            const double2 c = s_u[t * NK + (kz + K)];
            const double2 p = cmul(make_double2(alpha * c.x, alpha * c.y), twiddle(twz, kz * z, nz, +1));
            s.x += p.x;
            s.y += p.y;
        }
        s_g[t] = s;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < nr * NH; t += SF_BLOCK) {
        const int r = t / NH, ck = t - r * NH, y = y0 + r;  // ck = c (K + 1) + kx
        double2 s = make_double2(0.0, 0.0);
        for (int ky = -K; ky <= K; ky++) {
            const double2 p = cmul(s_g[ck * NK + (ky + K)], twiddle(twy, ky * y, ny, +1));
            s.x += p.x;
            s.y += p.y;
        }
        s_h[r][ck] = s;
    }
    __syncthreads();
    double* const f[3] = {fx, fy, fz};
    for (int x = threadIdx.x & 63; x < nx; x += 64) {
        double2 w[K + 1];
#pragma unroll
        for (int k = 1; k <= K; k++) w[k] = twiddle(twx, k * x, nx, +1);
        for (int r = threadIdx.x >> 6; r < nr; r += W) {
            const long s = ((long)z * ny + y0 + r) * px + x;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                double v = s_h[r][c * (K + 1)].x;
#pragma unroll
                for (int k = 1; k <= K; k++) {
                    const double2 h = s_h[r][c * (K + 1) + k];
                    v += 2.0 * (h.x * w[k].x - h.y * w[k].y);
                }
                f[c][s] = v;
            }
        }
    }
}

template <int K, typename T>
hipError_t spectral_k(const SpectralWork& w, const Grid& G, int k2lo, int k2hi, int band, double eps,
                      const T* u1, const T* u2, const T* u3, double* fx, double* fy, double* fz, hipStream_t st) {
    constexpr int NK = 2 * K + 1, NB = 3 * (K + 1) * NK;
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    const long rows = (long)ny * nz;
    constexpr int RPB = SF_BLOCK / 64 * RF_ROWS;
    hipLaunchKernelGGL((sf_rows_fwd<K, T>), dim3((rows + RPB - 1) / RPB), dim3(SF_BLOCK), 0, st, nx, G.px, ny, nz, u1,
                       u2, u3, w.twx, w.A);
    constexpr int NC = NB * NK, WPB = SF_BLOCK / 64;
    hipLaunchKernelGGL((sf_cols_fwd<K>), dim3((nz * NB + WPB - 1) / WPB), dim3(SF_BLOCK), 0, st, ny, nz, w.A, w.twy,
                       w.B);
    hipLaunchKernelGGL((sf_zsum<K>), dim3((NC + WPB - 1) / WPB), dim3(SF_BLOCK), 0, st, nx, ny, nz, w.B, w.twz, w.C);
    const int chunks = (ny + SF_ROWS - 1) / SF_ROWS;
    hipLaunchKernelGGL((sf_force<K>), dim3((unsigned)chunks * nz), dim3(SF_BLOCK), 0, st, nx, G.px, ny, nz, k2lo, k2hi,
                       band, eps, w.C, w.twx, w.twy, w.twz, w.elow, fx, fy, fz);
    return hipGetLastError();
}

// modes |k_a| <= kc - 1 transformed; kept: k2lo <= |k|^2 < k2hi
template <typename T>
hipError_t spectral_dispatch(const SpectralWork& w, const Grid& G, int kc, int k2lo, int k2hi, int band,
                             double eps, const T* u1, const T* u2, const T* u3, double* fx, double* fy, double* fz,
                             hipStream_t st) {
    switch (kc - 1) {
        case 1: return spectral_k<1, T>(w, G, k2lo, k2hi, band, eps, u1, u2, u3, fx, fy, fz, st);
        case 2: return spectral_k<2, T>(w, G, k2lo, k2hi, band, eps, u1, u2, u3, fx, fy, fz, st);
        case 3: return spectral_k<3, T>(w, G, k2lo, k2hi, band, eps, u1, u2, u3, fx, fy, fz, st);
        case 4: return spectral_k<4, T>(w, G, k2lo, k2hi, band, eps, u1, u2, u3, fx, fy, fz, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

size_t spectral_work_doubles(int nx, int ny, int nz, int kc) {
    const size_t K = (size_t)(kc - 1), NK = 2 * K + 1, NB = 3 * (K + 1) * NK;
    const size_t rows = (size_t)ny * nz;
    const size_t cplx = rows * 3 * (K + 1)      // A
                        + (size_t)nz * NB        // B
                        + NB * NK                // C
                        + (size_t)nx + ny + nz;  // twiddle tables
    return 2 * cplx + 1;                         // + E_low
}

void spectral_work_layout(SpectralWork& w, double* base, int nx, int ny, int nz, int kc) {
    const size_t K = (size_t)(kc - 1), NK = 2 * K + 1, NB = 3 * (K + 1) * NK;
    double2* p = reinterpret_cast<double2*>(base);
    w.A = p;
    p += (size_t)ny * nz * 3 * (K + 1);
    w.B = p;
    p += (size_t)nz * NB;
    w.C = p;
    p += NB * NK;
    w.twx = p;
    p += nx;
    w.twy = p;
    p += ny;
    w.twz = p;
    p += nz;
    w.elow = reinterpret_cast<double*>(p);
}

hipError_t launch_spectral_force(const SpectralWork& w, const Grid& G, int kc, double eps, const double* u1,
                                 const double* u2, const double* u3, double* fx, double* fy, double* fz,
                                 hipStream_t st) {
    return spectral_dispatch<double>(w, G, kc, 1, kc * kc, 0, eps, u1, u2, u3, fx, fy, fz, st);
}

hipError_t launch_spectral_force(const SpectralWork& w, const Grid& G, int kc, double eps, const float* u1,
                                 const float* u2, const float* u3, double* fx, double* fy, double* fz,
                                 hipStream_t st) {
    return spectral_dispatch<float>(w, G, kc, 1, kc * kc, 0, eps, u1, u2, u3, fx, fy, fz, st);
}

hipError_t launch_spectral_band(const SpectralWork& w, const Grid& G, int klo, int khi, const double* u1,
                                const double* u2, const double* u3, double* o1, double* o2, double* o3,
                                hipStream_t st) {
    return spectral_dispatch<double>(w, G, khi, klo * klo, khi * khi, 1, 0.0, u1, u2, u3, o1, o2, o3, st);
}

}  // namespace drp
