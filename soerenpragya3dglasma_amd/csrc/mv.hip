// MV-model initial conditions on the device, SU(3):
//   CollidingObjects::SetWilsonLines  SC/COLLIDINGOBJECTS/CollidingObjects.cpp:318-371
//     (SetChargeDensities :34-102, SolveLaplaceEquation :131-176, SetNewWilsonLines :179-226,
//      LongitudinalProfile :30-32)
//   InitialConditions::SingleSheet    SC/INITIALCONDITIONS/SUNCCURRENTS/RevSingleNucleus.cpp:7-210
//     with Dynamics::SUNc::EvolveRhoViaFourier SC/DYNAMICS/SUNcDynamics.cpp:275-350 and
//     CollidingObjects::SetWilsonLinesForFirstStep SC/COLLIDINGOBJECTS/CollidingObjects.cpp:377-411
//   the initial state of Simulation::Run  SC/Simulation.cpp:327-378 (collision) and of the left / right
//     single-nucleus drivers (SC/LeftNucleusSimulation.cpp:343-357, SC/RightNucleusSimulation.cpp:343-357).
//
// The reference walks z sequentially and solves one transverse slice at a time.  Here every transverse
// operation (charge, smoothing, Poisson solve) runs on all z slices at once as batched 2D FFTs; only the
// path-ordered Wilson-line product runs along z, in eight runs side by side where the plane alone does not fill the chip
// (scan_chunks), and not at all for the separable MV charge (k_sheet_sep).
//
// Work arrays (allocated for the call, freed at the end):
//   F     complex, F[(a*Nz + z)*P + y*Nx + x], a = colour 0..7 (the FFT layout)
//   rho   real,    rho[a*S + s]  (s = x + Nx*(y + Ny*z))
//   V     Wilson lines in the tiled matrix layout (18 planes)
#include <cmath>
#include <limits>
#include <vector>

#include "internal.h"
#include "adjoint.h"
#include "fft_lds.h"

namespace glasma {

namespace {

struct Wk {
    double* F = nullptr;
    double* rho = nullptr;
    double* V = nullptr;
    double* xi = nullptr;
};

__device__ __forceinline__ long fidx(const Geom& g, int a, long s) {
    // complex entry (a, s) of F; s = s2 + P*z so (a*Nz + z)*P + s2 = a*S + s
    return (long)a * g.S + s;
}

__device__ __forceinline__ double psqr2(const Geom& g, int px, int py, double ax, double ay) {
    return (2.0 - 2.0 * cos(2.0 * kPi * px / (double)g.nx)) / (ax * ax) +
           (2.0 - 2.0 * cos(2.0 * kPi * py / (double)g.ny)) / (ay * ay);
}

// SetChargeDensities: rho(z) = mult * sqrt(ax ay) * T(z) * xi with T the unit-area Gaussian in index units
__global__ void k_charge(double* __restrict__ F, const double* __restrict__ xi, Geom g, double mult_norm,
                         int center, double width) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const int z = (int)(s / g.P);
    const long s2 = s - (long)z * g.P;
    const double u = (z - center) / width;
    const double prof = exp(-0.5 * u * u) / sqrt(2.0 * kPi * width * width);
    const double c = mult_norm * prof;
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        F[2 * i] = c * xi[a + 8 * s2];
        F[2 * i + 1] = 0.0;
    }
}

// momentum-space factors of one z slice batch.  mode 0: smoothing nf * exp(-p^2/2 Lambda^2) p^2/(p^2+m^2);
// mode 1: Poisson nf / p^2 with the zero mode set to 0.
__global__ void k_transverse_filter(double* __restrict__ F, Geom g, double ax, double ay, double lam, double meff,
                                   int mode) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const long s2 = s % g.P;
    const int px = (int)(s2 % g.nx), py = (int)(s2 / g.nx);
    const double p2 = psqr2(g, px, py, ax, ay);
    const double nf = 1.0 / ((double)g.nx * g.ny);
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        double re = F[2 * i], im = F[2 * i + 1];
        if (mode == 0) {
            const double f = exp(-p2 / (2.0 * lam * lam));
            re = nf * re * f * p2 / (p2 + meff * meff);
            im = nf * im * f * p2 / (p2 + meff * meff);
        } else if (px == 0 && py == 0) {
            re = 0.0;
            im = 0.0;
        } else {
            re = nf * re / p2;
            im = nf * im / p2;
        }
        F[2 * i] = re;
        F[2 * i + 1] = im;
    }
}

// rho = Re F (optional), then F = (Re F, 0)
__global__ void k_take_real(double* __restrict__ F, double* __restrict__ rho, Geom g) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        if (rho) rho[(long)a * g.S + s] = F[2 * i];
        F[2 * i + 1] = 0.0;
    }
}

// F = (rho, 0)
__global__ void k_load_real(double* __restrict__ F, const double* __restrict__ rho, Geom g) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        F[2 * i] = rho[(long)a * g.S + s];
        F[2 * i + 1] = 0.0;
    }
}

// SetNewWilsonLines for all z in the reference's order (L: Nz-1 down to 0 with exp(-i A t / sqrt 2); R: 0 up to Nz-1
// with exp(+i A t / sqrt 2)): W <- exp(+-i A(z) t / sqrt 2) W, V(z) = W.  The product is cut into runs of z,
// one wave each, for the block's 64 transverse sites: a run's partial products, then, from the runs' totals in LDS, the
// product of all earlier runs multiplied in.  One thread per site walking all of z is a serial chain of Nz exponentials on
// a chip with P / 64 waves: 170 us at 48 x 48 x 128, in eight runs 85.  The runs read and write V once more, so large
// planes, whose waves fill the chip, take one: 128 x 128 x 256 404 us with one and 375 with eight, 256 x 256 x 128 472
// and 882.
constexpr int kScanChunks = 8;
int scan_chunks(const Geom& g) { return g.P <= 16384 ? kScanChunks : 1; }
size_t scan_lds(int chunks) { return sizeof(double) * chunks * 18 * 64; }
__device__ __forceinline__ void st_end(double* ends, int c, const M3& A) {
    double* const q = ends + (size_t)c * 18 * 64 + (threadIdx.x & 63);
#pragma unroll
    for (int k = 0; k < 9; k++) {
        q[128 * k] = A.re[k];
        q[128 * k + 64] = A.im[k];
    }
}
__device__ __forceinline__ void ld_end(const double* ends, int c, M3& A) {
    const double* const q = ends + (size_t)c * 18 * 64 + (threadIdx.x & 63);
#pragma unroll
    for (int k = 0; k < 9; k++) {
        A.re[k] = q[128 * k];
        A.im[k] = q[128 * k + 64];
    }
}
__global__ void __launch_bounds__(64 * kScanChunks) k_wilson_scan(const double* __restrict__ F, double* __restrict__ V,
                                                                  Geom g, int right) {
    extern __shared__ double ends[];
    const int nc = blockDim.x >> 6, c = threadIdx.x >> 6, len = (g.nz + nc - 1) / nc;
    const long s2 = (long)blockIdx.x * 64 + (threadIdx.x & 63);
    const int k0 = min(g.nz, c * len), k1 = s2 < g.P ? min(g.nz, k0 + len) : k0;
    M3 W, X, T;
    set_unit(W);
    const double cf = (right ? 1.0 : -1.0) / kSqrt2;
    for (int k = k0; k < k1; k++) {
        const int z = right ? k : g.nz - 1 - k;
        const long s = s2 + g.P * z;
        double col[8];
        for (int a = 0; a < 8; a++) col[a] = F[2 * fidx(g, a, s)];
        expi(cf, col, X);
        mul_nn(X, W, T);
        W = T;
        stm<long>(V, kGPlanes, 0, s, W);
    }
    st_end(ends, c, W);
    __syncthreads();
    if (c == 0) return;
    ld_end(ends, 0, W);
    for (int j = 1; j < c; j++) {
        ld_end(ends, j, X);
        mul_nn(X, W, T);
        W = T;
    }
    for (int k = k0; k < k1; k++) {
        const long s = s2 + g.P * (right ? k : g.nz - 1 - k);
        ldm<long>(V, kGPlanes, 0, s, X);
        mul_nn(X, W, T);
        stm<long>(V, kGPlanes, 0, s, T);
    }
}

// transverse links V^dag(x) V(x + mu) for mu = x, y and the unit z link, for z in [zlo, zhi]
__global__ void k_sheet_links(const double* __restrict__ V, double* __restrict__ U, Geom g, int zlo, int zhi) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long n = (long)(zhi - zlo + 1) * g.P;
    if (i >= n) return;
    const long s = i + (long)zlo * g.P;
    const int z = (int)(s / g.P);
    const long s2 = s - (long)z * g.P;
    const int x = (int)(s2 % g.nx), y = (int)(s2 / g.nx);
    M3 A, B, C;
    ldm<long>(V, kGPlanes, 0, s, A);
    ldm<long>(V, kGPlanes, 0, sidx(g, x + 1, y, z), B);
    mul_dn(A, B, C);
    stm<long>(U, kUPlanes, 0, s, C);
    ldm<long>(V, kGPlanes, 0, sidx(g, x, y + 1, z), B);
    mul_dn(A, B, C);
    stm<long>(U, kUPlanes, 18, s, C);
    set_unit(C);
    stm<long>(U, kUPlanes, 36, s, C);
}

// EvolveRhoViaFourier phase: F(pz) *= nf * exp(i sgn omega(pz) dt), sgn by half-spectrum and direction
__global__ void k_evolve_phase(double* __restrict__ F, Geom g, double az, double dt, int right) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const int pz = (int)(s / g.P);
    const double om = sqrt((2.0 - 2.0 * cos(2.0 * kPi * (double)pz / (double)g.nz)) / (az * az));
    double sgn;
    if (!right) sgn = (pz < g.nz / 2) ? -1.0 : 1.0;
    else sgn = (pz < g.nz / 2) ? 1.0 : -1.0;
    double sn, cs;
    sincos(sgn * om * dt, &sn, &cs);
    const double nf = 1.0 / g.nz;
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        const double re = nf * F[2 * i], im = nf * F[2 * i + 1];
        F[2 * i] = cs * re - sn * im;
        F[2 * i + 1] = sn * re + cs * im;
    }
}

// One sheet (nucleus) of an initial state: its direction, the z range [zlo, zhi] of its fields, the plane groups of J
// that take its J-stat and J, and, for the separable MV charge, the factors of c(z).
struct SheetSide {
    int right, zlo, zhi, wstat, wj;
    int center;
    double width, mult_norm;
};
struct SheetSides {
    SheetSide s[2];
    int n;
};
SheetSide sheet_side(bool right, int zlo, int zhi, int wstat, int wj) {
    return SheetSide{right ? 1 : 0, zlo, zhi, wstat, wj, 0, 1.0, 0.0};
}

// The separable MV charge rho(x, y, z) = c(z) xi(x, y).  Its work array, for n sides with two colours to a complex
// entry (the filters are real and even in p, so they act on the real and the imaginary part alike):
//   A    [side][pair][P] complex: xi on the way in, then the potential's transverse factor a(x, y)
//   prof [side][5 nz]: the evolved transform of c (2 nz), c evolved by dt (nz), and the partial sums of c and of c
//        evolved from the side the scan starts on up to and including z (nz each)
__device__ __forceinline__ double mv_profile(const SheetSide& sd, int z) {
    const double u = (z - sd.center) / sd.width;
    return sd.mult_norm * (exp(-0.5 * u * u) / sqrt(2.0 * kPi * sd.width * sd.width));  // k_charge's factor
}
// smoothing x Poisson over one transverse round trip: nf exp(-p^2/2 Lambda^2) p^2/(p^2+m^2) / p^2, the zero mode 0
__device__ __forceinline__ double sheet_filter(const Geom& g, int px, int py, double ax, double ay, double lam,
                                               double meff) {
    if (px == 0 && py == 0) return 0.0;
    const double p2 = psqr2(g, px, py, ax, ay);
    const double nf = 1.0 / ((double)g.nx * g.ny);
    const double fs = nf * exp(-p2 / (2.0 * lam * lam)) * p2 / (p2 + meff * meff);
    return fs / p2;
}

// coefficient pz of the side's profile evolved by dt: sum_z c(z) e^{-2 pi i pz z / nz} times k_evolve_phase's factor.
// One wave per output; the terms are dealt to the lanes.
__device__ __forceinline__ void profile_dft(double* __restrict__ prof, const SheetSide& sd, int nz, int pz, double az,
                                            double dt) {
    const int lane = threadIdx.x & 63;
    double re = 0.0, im = 0.0;
    for (int z = lane; z < nz; z += 64) {
        double sn, cs;
        sincos(-2.0 * kPi * (double)(((unsigned)pz * (unsigned)z) % (unsigned)nz) / (double)nz, &sn, &cs);
        const double c = mv_profile(sd, z);
        re = fma(c, cs, re);
        im = fma(c, sn, im);
    }
    re = wave_sum(re);
    im = wave_sum(im);
    const double om = sqrt((2.0 - 2.0 * cos(2.0 * kPi * (double)pz / (double)nz)) / (az * az));
    double sgn;
    if (!sd.right) sgn = (pz < nz / 2) ? -1.0 : 1.0;
    else sgn = (pz < nz / 2) ? 1.0 : -1.0;
    double sp, cp;
    sincos(sgn * om * dt, &sp, &cp);
    if (lane == 0) {
        prof[2 * pz] = cp * re - sp * im;
        prof[2 * pz + 1] = sp * re + cp * im;
    }
}

// Blocks [0, 4 planes): the transverse factor of one pair of colours, xi -> a(x, y), both transforms and the filter in
// LDS (two buffers of ny rows of ld entries, then the twiddles of nx and ny).  Every further wave: one coefficient of a
// side's evolved profile.  The two do not depend on each other and each alone leaves the chip nearly empty.
// What bounds this kernel is the chain of LDS stages of its one block per pair: 11 us at 16 x 16 x 32, where the separate
// passes (load, 4 transform launches, filter, 3 profile launches, the profiles' sums by one thread per output) took 70 us
// and their gaps, and 37 us for two nuclei of 64 x 64, where load, transforms and filter took 74 us.
// ODD: the odd primes of nx and ny (stockham).  Compiled for all of them it took 43.6 us at 64 x 64, without 37.0.
constexpr int kPlaneThreads = 512;
template <int ODD>
__global__ void __launch_bounds__(kPlaneThreads) k_sheet_plane(const double* __restrict__ xi, dbl2* __restrict__ A,
                                                               double* __restrict__ prof, Geom g, SheetSides sides,
                                                               int planes, int ld, Radices Rx, Radices Ry,
                                                               const dbl2* __restrict__ twx,
                                                               const dbl2* __restrict__ twy, double ax, double ay,
                                                               double az, double lam, double meff, double dt) {
    extern __shared__ dbl2 lds[];
    if ((int)blockIdx.x >= 4 * planes) {
        const int u = ((int)blockIdx.x - 4 * planes) * (kPlaneThreads / 64) + (int)(threadIdx.x >> 6);
        if (u >= sides.n * g.nz) return;
        const int side = u / g.nz;
        profile_dft(prof + (long)side * 5 * g.nz, sides.s[side], g.nz, u - side * g.nz, az, dt);
        return;
    }
    const int side = blockIdx.x >> 2, pair = blockIdx.x & 3;  // as in A
    const int P = (int)g.P, bs = g.ny * ld;
    dbl2* const tx = lds + 2 * bs;
    dbl2* const ty = tx + g.nx;
    for (int k = threadIdx.x; k < g.nx; k += kPlaneThreads) tx[k] = twx[k];
    for (int k = threadIdx.x; k < g.ny; k += kPlaneThreads) ty[k] = twy[k];
    const double* const src = xi + 8 * g.P * side + 2 * pair;
    const float rnx = 1.0f / (float)g.nx;
    for (int i = threadIdx.x; i < P; i += kPlaneThreads) {
        const int y = qdiv(i, g.nx, rnx);
        lds[y * ld + i - y * g.nx] = dbl2{src[8 * i], src[8 * i + 1]};
    }
    __syncthreads();
    int cur = stockham<false, ODD>(lds, bs, 0, Rx, g.ny, ld, -1, tx);
    cur = stockham<false, ODD>(lds, bs, cur, Ry, g.nx, 1, -1, ty, ld);
    for (int i = threadIdx.x; i < P; i += kPlaneThreads) {
        const int y = qdiv(i, g.nx, rnx), x = i - y * g.nx;
        lds[cur * bs + y * ld + x] *= sheet_filter(g, x, y, ax, ay, lam, meff);
    }
    __syncthreads();
    cur = stockham<false, ODD>(lds, bs, cur, Ry, g.nx, 1, +1, ty, ld);
    cur = stockham<false, ODD>(lds, bs, cur, Rx, g.ny, ld, +1, tx);
    for (int i = threadIdx.x; i < P; i += kPlaneThreads) {
        const int y = qdiv(i, g.nx, rnx);
        A[(long)blockIdx.x * g.P + i] = lds[cur * bs + y * ld + i - y * g.nx];
    }
}

// the same in separate passes, for planes beyond the LDS: A = xi with two colours to an entry, and the filter
__global__ void k_sheet_load(const double* __restrict__ xi, dbl2* __restrict__ A, long P, int n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 4 * P * n) return;
    const long q = i / P, s2 = i - q * P;
    const double* const src = xi + 8 * (P * (q >> 2) + s2) + 2 * (q & 3);
    A[i] = dbl2{src[0], src[1]};
}
__global__ void k_sheet_filter(dbl2* __restrict__ A, Geom g, int ncomp, double ax, double ay, double lam, double meff) {
    const long s2 = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s2 >= g.P) return;
    const int px = (int)(s2 % g.nx), py = (int)(s2 / g.nx);
    const double f = sheet_filter(g, px, py, ax, ay, lam, meff);
    for (int a = 0; a < ncomp; a++) A[a * g.P + s2] *= f;
}

// c evolved by dt: the real part of the inverse transform of profile_dft's coefficients.  One wave per z of a side.
__global__ void __launch_bounds__(256) k_profile_evolve(double* __restrict__ prof, int nz, int n) {
    const int u = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (u >= n * nz) return;
    const int side = u / nz, z = u - side * nz;
    double* const pr = prof + (long)side * 5 * nz;
    double acc = 0.0;
    for (int pz = lane; pz < nz; pz += 64) {
        double sn, cs;
        sincos(2.0 * kPi * (double)(((unsigned)pz * (unsigned)z) % (unsigned)nz) / (double)nz, &sn, &cs);
        acc += pr[2 * pz] * cs - pr[2 * pz + 1] * sn;
    }
    acc = wave_sum(acc);
    if (lane == 0) pr[2 * nz + z] = acc / nz;
}
// partial sums of c and c evolved in the order of the Wilson lines (left sheet: from Nz - 1 down, right: from 0 up).
// One block per side: each thread sums a run, the runs' sums are scanned in LDS.
__global__ void __launch_bounds__(256) k_profile_sums(double* __restrict__ prof, int nz, SheetSides sides) {
    __shared__ double part[2][2][256];
    const SheetSide sd = sides.s[blockIdx.x];
    double* const pr = prof + (long)blockIdx.x * 5 * nz;
    const int t = threadIdx.x, m = (nz + 255) / 256, k0 = min(nz, t * m), k1 = min(nz, k0 + m);
    double s0 = 0.0, s1 = 0.0;
    for (int k = k0; k < k1; k++) {
        const int z = sd.right ? k : nz - 1 - k;
        s0 += mv_profile(sd, z);
        s1 += pr[2 * nz + z];
    }
    int b = 0;
    part[0][0][t] = s0;
    part[0][1][t] = s1;
    __syncthreads();
    for (int o = 1; o < 256; o <<= 1, b ^= 1) {
        part[b ^ 1][0][t] = part[b][0][t] + (t >= o ? part[b][0][t - o] : 0.0);
        part[b ^ 1][1][t] = part[b][1][t] + (t >= o ? part[b][1][t - o] : 0.0);
        __syncthreads();
    }
    s0 = t ? part[b][0][t - 1] : 0.0;
    s1 = t ? part[b][1][t - 1] : 0.0;
    for (int k = k0; k < k1; k++) {
        const int z = sd.right ? k : nz - 1 - k;
        s0 += mv_profile(sd, z);
        s1 += pr[2 * nz + z];
        pr[3 * nz + z] = s0;
        pr[4 * nz + z] = s1;
    }
}

// The sheet's U(t + dt), UOld and E(t + dt/2) from the separable potentials A0 = c(z) a(x, y) and A1 = c_ev(z) a(x, y).
// The exponents of one transverse site along z are multiples of one matrix a(x, y) and commute, so the path-ordered
// product of SetNewWilsonLines is one exponential, V(z) = exp(+-i a(x, y) / sqrt 2 * sum of c over the layers passed):
// no serial chain in z, and no Wilson line is stored; each thread forms the four lines its link and its logarithm need.
// One thread per site and transverse direction (blockIdx.y = 2 side + mu).  Bound by the exponentials and the Jacobi
// sweeps of the logarithm.  The scans (one thread per transverse site walking z), the link passes and the E pass it
// replaces took 97 us at 16 x 16 x 32 (60 of them the scans' serial chain), where this takes 23, and for two nuclei
// 1490 us at 64 x 64 x 256 (534) and 22.2 ms at 256 x 256 x 512 (18.1).
__global__ void __launch_bounds__(256) k_sheet_sep(const dbl2* __restrict__ A, const double* __restrict__ prof,
                                                   double* __restrict__ U, double* __restrict__ UO,
                                                   double* __restrict__ E, Geom g, SheetSides sides, double coff0,
                                                   double coff1) {
    const int side = blockIdx.y >> 1, mu = blockIdx.y & 1;
    const SheetSide& sd = sides.s[side];
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)(sd.zhi - sd.zlo + 1) * g.P) return;
    const long s = i + (long)sd.zlo * g.P;
    const int z = (int)(s / g.P);
    const long s2 = s - (long)z * g.P;
    const int x = (int)(s2 % g.nx), y = (int)(s2 / g.nx);
    const long sn = mu == 0 ? sidx(g, x + 1, y, 0) : sidx(g, x, y + 1, 0);
    const dbl2* const Ap = A + 4 * g.P * side;
    double a[8], b[8];
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const dbl2 v = Ap[p * g.P + s2], w = Ap[p * g.P + sn];
        a[2 * p] = v.x;
        a[2 * p + 1] = v.y;
        b[2 * p] = w.x;
        b[2 * p + 1] = w.y;
    }
    const double* const sums = prof + (long)side * 5 * g.nz + 3 * g.nz;
    const double c = (sd.right ? 1.0 : -1.0) / kSqrt2;
    M3 V, W, L[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const double f = c * sums[t * g.nz + z];
        expi(f, a, V);
        expi(f, b, W);
        mul_dn(V, W, L[t]);
        stm<long>(t ? U : UO, kUPlanes, 18 * mu, s, L[t]);
    }
    set_unit(V);
    stm<long>(mu == 0 ? U : UO, kUPlanes, 36, s, V);
    mul_nd(L[1], L[0], V);
    double e[8];
    ilog(mu == 0 ? coff0 : coff1, V, e);
    stv<long>(E, kEPlanes, 8 * mu, s, e);
    if (mu == 0) {
        double zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        stv<long>(E, kEPlanes, 16, s, zero);
    }
}

// E_perp(t + dt/2) = MatrixILog(coff_mu, U_mu UOld_mu^dag), E_z = 0 for z in [zlo, zhi]  (:66-92).  Up to 2^19 sites
// each direction has threads of its own (efield_grid): 8.6 us against 11.6 at 32 x 32 x 32, 106 against 126 at
// 48 x 48 x 128, but 312 against 291 at 128 x 128 x 128, where one direction's threads fill the chip.
__global__ void __launch_bounds__(256) k_sheet_efield(const double* __restrict__ U, const double* __restrict__ UO, double* __restrict__ E,
                               Geom g, int zlo, int zhi, double coff0, double coff1) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long n = (long)(zhi - zlo + 1) * g.P;
    if (i >= n) return;
    const long s = i + (long)zlo * g.P;
    for (int mu = blockIdx.y; mu < 2; mu += gridDim.y) {
        M3 A, B, C;
        ldm<long>(U, kUPlanes, 18 * mu, s, A);
        ldm<long>(UO, kUPlanes, 18 * mu, s, B);
        mul_nd(A, B, C);
        double e[8];
        ilog(mu == 0 ? coff0 : coff1, C, e);
        stv<long>(E, kEPlanes, 8 * mu, s, e);
    }
    if (blockIdx.y) return;
    double zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    stv<long>(E, kEPlanes, 16, s, zero);
}

// J_stat = sqrt2 * sum_{i=x,y} (E_i(x) - U_i^dag(x-i) E_i(x-i) U_i(x-i)) inside [zlo, zhi], 0 outside
// (:98-125), of the side blockIdx.y.
__global__ void __launch_bounds__(256) k_sheet_jstat(const double* __restrict__ U, const double* __restrict__ E,
                                                     double* __restrict__ J, Geom g, SheetSides A) {
    const int zlo = A.s[blockIdx.y].zlo, zhi = A.s[blockIdx.y].zhi, wstat = A.s[blockIdx.y].wstat;
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const int z = (int)(s / g.P);
    const long s2 = s - (long)z * g.P;
    const int x = (int)(s2 % g.nx), y = (int)(s2 / g.nx);
    double js[8];
    if (z >= zlo && z <= zhi) {
        const long sx = sidx(g, x - 1, y, z);
        const long sy = sidx(g, x, y - 1, z);
        M3 Ux, Uy;
        double ex[8], ey[8], exm[8], eym[8], xd[8], yd[8];
        ldm<long>(U, kUPlanes, 0, sx, Ux);
        ldm<long>(U, kUPlanes, 18, sy, Uy);
        ldv<long>(E, kEPlanes, 0, s, ex);
        ldv<long>(E, kEPlanes, 8, s, ey);
        ldv<long>(E, kEPlanes, 0, sx, exm);
        ldv<long>(E, kEPlanes, 8, sy, eym);
        inv_adj_mul(Ux, exm, xd);
        inv_adj_mul(Uy, eym, yd);
        for (int a = 0; a < 8; a++) js[a] = kSqrt2 * ((ex[a] - xd[a]) + (ey[a] - yd[a]));
    } else {
        for (int a = 0; a < 8; a++) js[a] = 0.0;
    }
    stv<long>(J, kJPlanes, 8 * wstat, s, js);
}

// continuity inversion in z momentum space (:131-209):
//   J~(0) = J~stat(0); J~(N/2) = 0; otherwise J~ = J~stat (e^{-+ i omega dt} - 1) / (dt pZD)
// (conj = 1: the complex-conjugate filter, i.e. the transpose of the real-linear map)
__global__ void k_jinv(double* __restrict__ F, Geom g, double az, double dt, int right, int conj) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const int pz = (int)(s / g.P);
    const int nz = g.nz;
    const double om = sqrt((2.0 - 2.0 * cos(2.0 * kPi * (double)pz / (double)nz)) / (az * az));
    double es, ec;
    sincos(-2.0 * kPi * (double)pz / (double)nz, &es, &ec);
    // pZD = +-(1 - e)/az
    double zr = (1.0 - ec) / az, zi = -es / az;
    double sp, cp, sm, cm;
    sincos(om * dt, &sp, &cp);
    sincos(-om * dt, &sm, &cm);
    double pr, pi_, nr, ni;  // pNpos, pNneg
    if (right) {
        pr = cp - 1.0; pi_ = sp; nr = cm - 1.0; ni = sm;
    } else {
        zr = -zr; zi = -zi;
        pr = cm - 1.0; pi_ = sm; nr = cp - 1.0; ni = sp;
    }
    if (conj) {
        zi = -zi;
        pi_ = -pi_;
        ni = -ni;
    }
    const double dr = dt * zr, di = dt * zi;  // dt * pZD
    const double den = dr * dr + di * di;
    const double nf = 1.0 / nz;
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        const double jr = nf * F[2 * i], ji = nf * F[2 * i + 1];
        double outr, outi;
        if (pz == 0) {
            outr = jr; outi = ji;
        } else if (pz == nz / 2) {
            outr = 0.0; outi = 0.0;
        } else {
            const double mr = (pz < nz / 2) ? pr : nr, mi = (pz < nz / 2) ? pi_ : ni;
            // (j * m) / d
            const double qr = jr * mr - ji * mi, qi = jr * mi + ji * mr;
            outr = (qr * dr + qi * di) / den;
            outi = (qi * dr - qr * di) / den;
        }
        F[2 * i] = outr;
        F[2 * i + 1] = outi;
    }
}

// factor pz of k_jinv, 1/Nz included
__device__ __forceinline__ dbl2 jinv_factor(int pz, int nz, double az, double dt, int right) {
    const double nf = 1.0 / nz;
    if (pz == 0) return dbl2{nf, 0.0};
    if (pz == nz / 2) return dbl2{0.0, 0.0};
    const double om = sqrt((2.0 - 2.0 * cos(2.0 * kPi * (double)pz / (double)nz)) / (az * az));
    double es, ec, sp, cp;
    sincos(-2.0 * kPi * (double)pz / (double)nz, &es, &ec);
    sincos(om * dt, &sp, &cp);
    // the two branches of k_jinv: e^{+i om dt} - 1 for the lower half of the right sheet's spectrum and the upper
    // half of the left's, its conjugate otherwise
    const double mr = cp - 1.0, mi = (right != 0) == (pz < nz / 2) ? sp : -sp;
    const double sg = right ? 1.0 : -1.0;
    const double dr = dt * (sg * (1.0 - ec) / az), di = dt * (-sg * es / az);
    const double den = dr * dr + di * di;
    return dbl2{nf * ((mr * dr + mi * di) / den), nf * ((mi * dr - mr * di) / den)};
}

// J from J-stat: the continuity inversion (k_jinv between a forward and an inverse z transform, the real part kept) in
// one pass over the current field.  A tiled plane pair holds colours 2p and 2p + 1 of a site side by side, so a z line
// of a pair is read as one complex line: the map takes real lines to real lines once its factors are made Hermitian,
// h(k) = (H(k) + conj H(Nz - k)) / 2, which is what keeping the real part does.  blockIdx.y = side; a side's lines are
// taken lpb neighbours at a time by walking blocks, XCD k owning the k-th eighth of the groups.
// LDS: two buffers of lpb * ld entries, the two-level twiddles, h(k) for k <= Nz / 2.
// Separate passes (J-stat copied to a complex array, transform, factors, transform, real parts to J) moved 960 bytes a
// site beyond the J-stat itself; this one moves 128.  Two nuclei at 64 x 64 x 256: 318 us before, 147 now; at
// 256 x 256 x 512 12.6 and 5.2 ms (the LDS stages; the bytes alone would take 1.4).
// ODD: the odd primes of nz (stockham).  Compiled for all of them it took 161 us at 64 x 64 x 256 and 5.66 ms at 256 x 256
// x 512, without 143 us and 5.19 ms.
template <int ODD>
__global__ void __launch_bounds__(256) k_sheet_jinv(double* __restrict__ J, Geom g, SheetSides sides, Radices R, int lpb,
                                                    int ld, const dbl2* __restrict__ twg, double az, double dt) {
    extern __shared__ dbl2 lds[];
    const int n = R.n, bs = lpb * ld;
    const SheetSide& sd = sides.s[blockIdx.y];
    dbl2* const tw = lds + 2 * bs;
    dbl2* const h = tw + split_entries(n);
    for (int k = threadIdx.x; k < split_entries(n); k += 256) tw[k] = twg[k];
    for (int k = threadIdx.x; k <= n / 2; k += 256) {
        const dbl2 a = jinv_factor(k, n, az, dt, sd.right);
        const dbl2 b = k ? jinv_factor(n - k, n, az, dt, sd.right) : a;
        h[k] = dbl2{0.5 * (a.x + b.x), 0.5 * (a.y - b.y)};
    }
    const int lg = __builtin_ctz(lpb);
    const long gpp = (g.P + lpb - 1) / lpb, groups = 4 * gpp;  // groups of a pair, and of the side
    const long per = (groups + 7) / 8, last = min(groups, (long)(blockIdx.x % 8 + 1) * per);
    for (long q = (blockIdx.x % 8) * per + blockIdx.x / 8; q < last; q += gridDim.x / 8) {
        const int pair = (int)(q / gpp);
        const long s0 = (q - pair * gpp) * lpb;
        for (int i = threadIdx.x; i < lpb * n; i += 256) {
            const int li = i & (lpb - 1), z = i >> lg;
            const long s2 = s0 + li;
            dbl2 v = dbl2{0.0, 0.0};
            if (s2 < g.P) v = ld2(J + lidx<long>(kJPlanes, 8 * sd.wstat + 2 * pair, s2 + g.P * z));
            lds[li * ld + z] = v;
        }
        __syncthreads();
        int cur = stockham<true, ODD>(lds, bs, 0, R, lpb, ld, -1, tw);
        for (int i = threadIdx.x; i < lpb * n; i += 256) {
            const int li = i & (lpb - 1), k = i >> lg;
            dbl2 f = h[2 * k <= n ? k : n - k];
            if (2 * k > n) f.y = -f.y;
            dbl2* const at = lds + cur * bs + li * ld + k;
            *at = cmul(f, *at);
        }
        __syncthreads();
        cur = stockham<true, ODD>(lds, bs, cur, R, lpb, ld, +1, tw);
        for (int i = threadIdx.x; i < lpb * n; i += 256) {
            const int li = i & (lpb - 1), z = i >> lg;
            const long s2 = s0 + li;
            const dbl2 v = lds[cur * bs + li * ld + z];
            if (s2 < g.P) *(dbl2*)(J + lidx<long>(kJPlanes, 8 * sd.wj + 2 * pair, s2 + g.P * z)) = v;
        }
        __syncthreads();
    }
}

// rho (real, a*S + s) -> host AoS with ghosts (a + 8*Index3D)
__global__ void k_rho_to_aos(const double* __restrict__ rho, double* __restrict__ out, Geom g) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 8 * g.S) return;
    const long s = i / 8;
    const int a = (int)(i % 8);
    out[i] = rho[(long)a * g.S + s];
}

inline dim3 grid1(long n) { return dim3((unsigned)((n + 255) / 256)); }
inline dim3 efield_grid(long n) { return dim3(grid1(n).x, n <= (1L << 19) ? 2 : 1); }

int alloc_work(glasma_ctx* ctx, Wk& w) {
    const long S = ctx->g.S, Sp = pad_sites(S);
    int rc = ensure_fftbuf(ctx, 16 * (size_t)S);
    if (rc) return rc;
    w.F = ctx->fftbuf;
    GL_HIP(ctx, hipMalloc(&w.rho, 8 * (size_t)S * sizeof(double)));
    GL_HIP(ctx, hipMalloc(&w.V, (size_t)kGPlanes * Sp * sizeof(double)));
    GL_HIP(ctx, hipMalloc(&w.xi, 8 * (size_t)ctx->g.P * sizeof(double)));
    return 0;
}
void free_work(Wk& w) {
    if (w.rho) (void)hipFree(w.rho);
    if (w.V) (void)hipFree(w.V);
    if (w.xi) (void)hipFree(w.xi);
    w = Wk();
}

#define GL_RC(x)                  \
    do {                          \
        int _rc = (x);            \
        if (_rc) return _rc;      \
    } while (0)
#define GL_FFT(ctx, x)                                                                       \
    do {                                                                                     \
        int _rc = (x);                                                                       \
        if (_rc) return set_error(ctx, _rc, std::string("FFT failed (lengths must be 2^a 3^b p <= 2048, " \
                                                        "prime factors <= 13): ") + fft_last_error()); \
    } while (0)

int wilson_scan(glasma_ctx* ctx, const double* F, double* V, int right) {
    const int nc = scan_chunks(ctx->g);
    // the runs' totals are above what a kernel gets without asking
    GL_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(&k_wilson_scan),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)scan_lds(kScanChunks)));
    hipLaunchKernelGGL(k_wilson_scan, dim3((unsigned)((ctx->g.P + 63) / 64)), dim3(64 * nc), scan_lds(nc), ctx->stream, F, V,
                       ctx->g, right);
    return 0;
}

// Poisson solve of every transverse slice: F (real parts) -> A, imaginary parts of the result dropped
int poisson_all(glasma_ctx* ctx, double* F) {
    const Geom& g = ctx->g;
    GL_FFT(ctx, fft_xy(ctx->stream, F, g, 8, g.nz, -1));
    hipLaunchKernelGGL(k_transverse_filter, grid1(g.S), dim3(256), 0, ctx->stream, F, g, ctx->p.a[0], ctx->p.a[1], 0.0,
                       0.0, 1);
    GL_FFT(ctx, fft_xy(ctx->stream, F, g, 8, g.nz, +1));
    return 0;
}

// the per-z part of CollidingObjects::SetWilsonLines for the charge held in F (real parts): smoothing
// (UV factor exp(-p^2 / 2 Lambda^2), 1 for Lambda = infinity; IR factor p^2 / (p^2 + m^2)), w.rho = the
// smoothed charge, Poisson solve and the path-ordered Wilson lines w.V
int wilson_from_charge(glasma_ctx* ctx, Wk& w, double lambda, double meff, bool right) {
    const Geom& g = ctx->g;
    GL_FFT(ctx, fft_xy(ctx->stream, w.F, g, 8, g.nz, -1));
    hipLaunchKernelGGL(k_transverse_filter, grid1(g.S), dim3(256), 0, ctx->stream, w.F, g, ctx->p.a[0], ctx->p.a[1],
                       lambda, meff, 0);
    GL_FFT(ctx, fft_xy(ctx->stream, w.F, g, 8, g.nz, +1));
    hipLaunchKernelGGL(k_take_real, grid1(g.S), dim3(256), 0, ctx->stream, w.F, w.rho, g);
    GL_RC(poisson_all(ctx, w.F));
    GL_RC(wilson_scan(ctx, w.F, w.V, right ? 1 : 0));
    GL_HIP(ctx, hipGetLastError());
    return 0;
}

// CollidingObjects::SetWilsonLines for one nucleus: w.rho = smoothed charge, w.V = Wilson lines
int set_wilson_lines(glasma_ctx* ctx, Wk& w, const glasma_mv_params* mv, const double* xi_host, bool right) {
    const Geom& g = ctx->g;
    GL_HIP(ctx, hipMemcpyAsync(w.xi, xi_host, 8 * (size_t)g.P * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    const double norm = std::sqrt(ctx->p.a[0] * ctx->p.a[1]);
    const double mult = right ? mv->nucleus_r : mv->nucleus_l;
    hipLaunchKernelGGL(k_charge, grid1(g.S), dim3(256), 0, ctx->stream, w.F, w.xi, g, mult * norm,
                       right ? mv->center_r : mv->center_l, right ? mv->sigma_r : mv->sigma_l);
    return wilson_from_charge(ctx, w, mv->lambda, mv->m_eff, right);
}

// J-stat from the transverse Gauss law and J from the z continuity inversion (RevSingleNucleus.cpp:98-209), all sides
int sheet_currents(glasma_ctx* ctx, const double* U, const double* E, double* J, const SheetSides& A) {
    const Geom& g = ctx->g;
    Radices R;
    GL_FFT(ctx, fft_radices(g.nz, R));
    const dbl2* tw = nullptr;
    GL_HIP(ctx, fft_twiddles_split(g.nz, &tw));
    size_t most = 0;
    GL_HIP(ctx, fft_lds_limit(&most));
    // lines per group: 64-byte rows (4) where three workgroups still fit a CU, else fewer.  The initial state took, at
    // 128 x 128 x 512, 6.5 to 7.2 ms with 2 lines (39 KiB) and 6.8 with 4 (75 KiB); at 128 x 128 x 1024 13.8 ms with 1
    // or 2 lines (42, 75 KiB) and 15.4 with 4 (one workgroup per CU).  A line of 2048 alone takes 84 KiB.
    int lpb = 4;
    auto bytes = [&](int l) {
        return sizeof(dbl2) * (2 * (size_t)l * (l > 1 ? g.nz + 1 : g.nz) + split_entries(g.nz) + g.nz / 2 + 1);
    };
    while (lpb > 1 && bytes(lpb) > 53 * 1024) lpb /= 2;
    const size_t lds = bytes(lpb);
    if (lds > most) return set_error(ctx, GLASMA_ERR_ARG, "the current's z line exceeds the LDS");
    const int odd = odd_level(R);
    const auto jinv = odd == 0 ? k_sheet_jinv<0> : odd == 1 ? k_sheet_jinv<1> : k_sheet_jinv<2>;
    if (lds > 65536)
        GL_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(jinv),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k_sheet_jstat, dim3(grid1(g.S).x, A.n), dim3(256), 0, ctx->stream, U, E, J, g, A);
    // blocks: at most 2048 a side, walking; a multiple of 8 for the XCD ranges
    const long groups = 4 * ((g.P + lpb - 1) / lpb);
    const unsigned blocks = (unsigned)(8 * std::min<long>(256, (groups + 7) / 8));
    hipLaunchKernelGGL(jinv, dim3(blocks, A.n), dim3(256), lds, ctx->stream, J, g, A, R, lpb,
                       lpb > 1 ? g.nz + 1 : g.nz, tw, ctx->p.a[2], ctx->p.dt);
    GL_HIP(ctx, hipGetLastError());
    return 0;
}

// InitialConditions::SingleSheet for one nucleus over [zlo, zhi]; J-stat into plane group wstat, J into w
int single_sheet(glasma_ctx* ctx, Wk& w, bool right, int zlo, int zhi, int wstat, int wj) {
    const Geom& g = ctx->g;
    const double dt = ctx->p.dt;
    double* U = ctx->U[ctx->cur];
    double* J = ctx->J[ctx->cur];
    const long nsl = (long)(zhi - zlo + 1) * g.P;
    // UOld = links of the sheet at t = 0 (:14-27)
    hipLaunchKernelGGL(k_sheet_links, grid1(nsl), dim3(256), 0, ctx->stream, w.V, ctx->UOld, g, zlo, zhi);
    // rho evolved by dt through the z FFT (:33, SUNcDynamics.cpp:275-350)
    hipLaunchKernelGGL(k_load_real, grid1(g.S), dim3(256), 0, ctx->stream, w.F, w.rho, g);
    GL_FFT(ctx, fft_z(ctx->stream, w.F, g, 8, -1));
    hipLaunchKernelGGL(k_evolve_phase, grid1(g.S), dim3(256), 0, ctx->stream, w.F, g, ctx->p.a[2], dt, right ? 1 : 0);
    GL_FFT(ctx, fft_z(ctx->stream, w.F, g, 8, +1));
    hipLaunchKernelGGL(k_take_real, grid1(g.S), dim3(256), 0, ctx->stream, w.F, (double*)nullptr, g);
    // Wilson lines of the evolved charge (SetWilsonLinesForFirstStep, no smoothing) and U(t + dt) (:40-60)
    GL_RC(poisson_all(ctx, w.F));
    GL_RC(wilson_scan(ctx, w.F, w.V, right ? 1 : 0));
    hipLaunchKernelGGL(k_sheet_links, grid1(nsl), dim3(256), 0, ctx->stream, w.V, U, g, zlo, zhi);
    // E(t + dt/2) from the logarithm of U UOld^dag (:66-92)
    const double acube = ctx->p.a[0] * ctx->p.a[1] * ctx->p.a[2];
    const double coff0 = -dt * ctx->p.a[0] * ctx->p.a[0] / acube;
    const double coff1 = -dt * ctx->p.a[1] * ctx->p.a[1] / acube;
    hipLaunchKernelGGL(k_sheet_efield, efield_grid(nsl), dim3(256), 0, ctx->stream, U, ctx->UOld, ctx->E, g, zlo, zhi, coff0,
                       coff1);
    // J-stat from the transverse Gauss law and J from the z continuity inversion (:98-209)
    SheetSides A;
    A.n = 1;
    A.s[0] = sheet_side(right, zlo, zhi, wstat, wj);
    return sheet_currents(ctx, U, ctx->E, J, A);
}

// CollidingObjects::SetWilsonLines and InitialConditions::SingleSheet for the MV nuclei of an initial state, using that
// the charge is separable, rho(x, y, z) = c(z) xi(x, y) (SetChargeDensities, k_charge).  The reference smooths the
// charge (a transverse round trip), solves Poisson (another), and for U(t + dt) evolves the smoothed charge along z (a z
// round trip) and solves Poisson again, taking real parts in between.  Those filters are linear and each acts on one set
// of axes, so both potentials factor: A0 = c(z) a(x, y) and A1 = c_ev(z) a(x, y), with a = the smoothing x Poisson of xi
// on one transverse slice and c_ev = the real part of c evolved by dt (the filters are real and even in p, so the real
// parts taken in between are exact up to round-off).  Links and E follow from these factors site by site
// (k_sheet_sep): no transform of the whole lattice and no scan in z.  All sides go through each launch together; their
// z ranges must not overlap.  m_eff = 0 keeps the separate steps (their smoothing factor is 0/0 at p = 0, which the
// reference's order spreads over the slice).  xi[side]: host arrays of 8 P doubles.
int mv_sheets(glasma_ctx* ctx, const glasma_mv_params* mv, SheetSides A, const double* const xi[2]) {
    const Geom& g = ctx->g;
    const double dt = ctx->p.dt;
    const double* a = ctx->p.a;
    const double norm = std::sqrt(a[0] * a[1]);
    long nmax = 0;
    for (int k = 0; k < A.n; k++) {
        SheetSide& sd = A.s[k];
        sd.center = sd.right ? mv->center_r : mv->center_l;
        sd.width = sd.right ? mv->sigma_r : mv->sigma_l;
        sd.mult_norm = (sd.right ? mv->nucleus_r : mv->nucleus_l) * norm;
        nmax = std::max(nmax, (long)(sd.zhi - sd.zlo + 1) * g.P);
    }
    Radices Rx, Ry, Rz;
    GL_FFT(ctx, fft_radices(g.nx, Rx));
    GL_FFT(ctx, fft_radices(g.ny, Ry));
    GL_FFT(ctx, fft_radices(g.nz, Rz));
    GL_RC(ensure_fftbuf(ctx, (size_t)A.n * (16 * (size_t)g.P + 5 * (size_t)g.nz)));
    dbl2* const F = reinterpret_cast<dbl2*>(ctx->fftbuf);
    double* const dxi = ctx->fftbuf + 8 * g.P * A.n;
    double* const prof = dxi + 8 * g.P * A.n;
    for (int k = 0; k < A.n; k++)
        GL_HIP(ctx, hipMemcpyAsync(dxi + 8 * g.P * k, xi[k], 8 * (size_t)g.P * sizeof(double), hipMemcpyHostToDevice,
                                   ctx->stream));
    // the transverse factor a(x, y) of each side: in one launch where a plane fits the LDS twice (up to about 70 x 70),
    // together with the profiles' transforms; else in separate passes
    size_t most = 0;
    GL_HIP(ctx, fft_lds_limit(&most));
    const int ld = g.nx | 1;
    const size_t need = sizeof(dbl2) * (2 * (size_t)g.ny * ld + g.nx + g.ny);
    const bool plane = need <= most;
    const dbl2 *twx = nullptr, *twy = nullptr;
    const int odd = plane ? std::max(odd_level(Rx), odd_level(Ry)) : 0;
    const auto sheet_plane = odd == 0 ? k_sheet_plane<0> : odd == 1 ? k_sheet_plane<1> : k_sheet_plane<2>;
    if (plane) {
        GL_HIP(ctx, fft_twiddles(g.nx, &twx));
        GL_HIP(ctx, fft_twiddles(g.ny, &twy));
        if (need > 65536)
            GL_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(sheet_plane),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)need));
    }
    const int planes = plane ? A.n : 0, wpb = kPlaneThreads / 64;
    hipLaunchKernelGGL(sheet_plane, dim3(4 * planes + (A.n * g.nz + wpb - 1) / wpb), dim3(kPlaneThreads),
                       plane ? need : 0, ctx->stream, dxi, F, prof, g, A, planes, ld, Rx, Ry, twx, twy, a[0], a[1], a[2],
                       mv->lambda, mv->m_eff, dt);
    if (!plane) {
        hipLaunchKernelGGL(k_sheet_load, grid1(4 * g.P * A.n), dim3(256), 0, ctx->stream, dxi, F, g.P, A.n);
        GL_FFT(ctx, fft_xy(ctx->stream, ctx->fftbuf, g, 4 * A.n, 1, -1));
        hipLaunchKernelGGL(k_sheet_filter, grid1(g.P), dim3(256), 0, ctx->stream, F, g, 4 * A.n, a[0], a[1], mv->lambda,
                           mv->m_eff);
        GL_FFT(ctx, fft_xy(ctx->stream, ctx->fftbuf, g, 4 * A.n, 1, +1));
    }
    hipLaunchKernelGGL(k_profile_evolve, dim3((A.n * g.nz + 3) / 4), dim3(256), 0, ctx->stream, prof, g.nz, A.n);
    hipLaunchKernelGGL(k_profile_sums, dim3(A.n), dim3(256), 0, ctx->stream, prof, g.nz, A);
    // U(t + dt) from A1 (SetWilsonLinesForFirstStep, :33-60), UOld from A0 (:14-27), E(t + dt/2) (:66-92)
    const double acube = a[0] * a[1] * a[2];
    double* U = ctx->U[ctx->cur];
    hipLaunchKernelGGL(k_sheet_sep, dim3(grid1(nmax).x, 2 * A.n), dim3(256), 0, ctx->stream, F, prof, U, ctx->UOld, ctx->E,
                       g, A, -dt * a[0] * a[0] / acube, -dt * a[1] * a[1] / acube);
    return sheet_currents(ctx, U, ctx->E, ctx->J[ctx->cur], A);
}

// ------------------------------------------------------------------------------------------------
// The left-moving sheet from a given charge density, with its intermediates kept, and the reverse-mode
// derivative of that map (cotangents of U, E, J+, J+stat at t = 0 -> cotangent of the charge density).
// Forward: rho_s = smooth(rho); A0 = poisson(rho_s); V0 = scan(A0); UOld = links(V0);
// rho_ev = evolve_L(rho_s); A1 = poisson(rho_ev); V1 = scan(A1); U = links(V1); E = ilog(U UOld^dag);
// J+stat = sqrt2 sum_i (E_i - Ad(U_i^dag(x-i)) E_i(x-i)); J+ = jinv_L(J+stat).
// The smoothing and Poisson filters are real and even in p (self-adjoint maps); the z-evolution and the
// current inversion transpose to their complex-conjugate filters (evolve_L^T = evolve_R).
// ------------------------------------------------------------------------------------------------
// F = (values of tiled planes p0..p0+7 of a field with NP planes, 0)
__global__ void k_load_planes(double* __restrict__ F, const double* __restrict__ X, Geom g, int NP, int p0) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        F[2 * i] = X[lidx<long>(NP, p0 + a, s)];
        F[2 * i + 1] = 0.0;
    }
}
// out[a*S + s] = x[a*S + s] + c * Re F
__global__ void k_axpy_real(double* __restrict__ out, const double* __restrict__ x, const double* __restrict__ F,
                            double c, Geom g) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 8 * g.S) return;
    out[i] = (x ? x[i] : 0.0) + c * F[2 * i];
}
__global__ void k_copy_real(double* __restrict__ out, const double* __restrict__ F, Geom g) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 8 * g.S) return;
    out[i] = F[2 * i];
}
__global__ void k_zero(double* __restrict__ p, long n) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// J+stat cotangent jsb (real, a*S + s) -> E_x, E_y and U_x, U_y cotangents (gathered at y from y + i)
__global__ void __launch_bounds__(256) k_ic_jstat_vjp(const double* __restrict__ U, const double* __restrict__ E,
                               const double* __restrict__ jsb, double* __restrict__ Ub, double* __restrict__ Eb,
                               Geom g) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const int z = (int)(s / g.P);
    const long s2 = s - (long)z * g.P;
    const int x = (int)(s2 % g.nx), y = (int)(s2 / g.nx);
    double own[8];
    for (int a = 0; a < 8; a++) own[a] = jsb[(long)a * g.S + s];
    for (int mu = 0; mu < 2; mu++) {
        const long sn = mu == 0 ? sidx(g, x + 1, y, z) : sidx(g, x, y + 1, z);
        double up[8], e[8], eb[8], t8[8];
        for (int a = 0; a < 8; a++) up[a] = jsb[(long)a * g.S + sn];
        M3 Um, Ubm;
        ldm<long>(U, kUPlanes, 18 * mu, s, Um);
        ldm<long>(Ub, kUPlanes, 18 * mu, s, Ubm);
        ldv<long>(E, kEPlanes, 8 * mu, s, e);
        ldv<long>(Eb, kEPlanes, 8 * mu, s, eb);
        adj_mul(Um, up, t8);
        for (int a = 0; a < 8; a++) eb[a] += kSqrt2 * own[a] - kSqrt2 * t8[a];
        acc_lvr(-kSqrt2, e, Um, up, Ubm);
        stv<long>(Eb, kEPlanes, 8 * mu, s, eb);
        stm<long>(Ub, kUPlanes, 18 * mu, s, Ubm);
    }
}

// 8x8 linear solve by Gaussian elimination with partial pivoting (A is overwritten); returns x in b
__device__ void solve8(double (&A)[8][8], double* b) {
    for (int c = 0; c < 8; c++) {
        int p = c;
        for (int r = c + 1; r < 8; r++)
            if (fabs(A[r][c]) > fabs(A[p][c])) p = r;
        if (p != c) {
            for (int k = 0; k < 8; k++) { const double t = A[c][k]; A[c][k] = A[p][k]; A[p][k] = t; }
            const double t = b[c]; b[c] = b[p]; b[p] = t;
        }
        const double inv = 1.0 / A[c][c];
        for (int r = c + 1; r < 8; r++) {
            const double f = A[r][c] * inv;
            for (int k = c; k < 8; k++) A[r][k] -= f * A[c][k];
            b[r] -= f * b[c];
        }
    }
    for (int c = 7; c >= 0; c--) {
        double v = b[c];
        for (int k = c + 1; k < 8; k++) v -= A[c][k] * b[k];
        b[c] = v / A[c][c];
    }
}

// E_mu = ilog(coff, M), M = U_mu UOld_mu^dag (mu = x, y): with A = i coff E t and the left-trivialised
// derivative G = sum_k (-ad_A)^k/(k+1)!, M^dag dM = G(i coff t dE); in components kappa = -2 Re tr(i t M^dag dM)
// = Ghat coff dE, so kappabar = Ghat^-T Ebar / coff and Mbar = 2 i M H(kappabar).  Ubar += Mbar UOld,
// UOldbar = Mbar^dag U.
__global__ void __launch_bounds__(256) k_ic_ilog_vjp(const double* __restrict__ U, const double* __restrict__ UO,
                              const double* __restrict__ E, const double* __restrict__ Eb, double* __restrict__ Ub,
                              double* __restrict__ UOb, Geom g, double coff0, double coff1) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    for (int mu = 0; mu < 2; mu++) {
        const double coff = mu == 0 ? coff0 : coff1;
        M3 Um, Uo, M;
        ldm<long>(U, kUPlanes, 18 * mu, s, Um);
        ldm<long>(UO, kUPlanes, 18 * mu, s, Uo);
        mul_nd(Um, Uo, M);
        double e[8], eb[8];
        ldv<long>(E, kEPlanes, 8 * mu, s, e);
        ldv<long>(Eb, kEPlanes, 8 * mu, s, eb);
        // row b = column b of Ghat: the coordinates (basis i t^a) of sum_k (-ad_A)^k (i t^b) / (k+1)!, A = i coff e^a t^a,
        // so -ad_A is ad_series' map with c = -coff
        double G[8][8];
        for (int b = 0; b < 8; b++) {
            double unit[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            unit[b] = 1.0;
            ad_series(-coff, e, unit, G[b]);
        }
        double kb[8];
        for (int a = 0; a < 8; a++) kb[a] = eb[a] / coff;
        solve8(G, kb);
        M3 Hk, Mb, T;
        herm_from_alg(1.0, kb, Hk);
        mul_nn(M, Hk, T);
        for (int k = 0; k < 9; k++) { Mb.re[k] = -2.0 * T.im[k]; Mb.im[k] = 2.0 * T.re[k]; }  // 2 i M H
        M3 Ubm, Ta;
        ldm<long>(Ub, kUPlanes, 18 * mu, s, Ubm);
        mul_nn(Mb, Uo, Ta);
        m3_axpy(1.0, Ta, Ubm);
        stm<long>(Ub, kUPlanes, 18 * mu, s, Ubm);
        mul_dn(Mb, Um, Ta);
        stm<long>(UOb, kUPlanes, 18 * mu, s, Ta);
    }
}

// V cotangent from the link cotangents of U_mu = V^dag(x) V(x + mu), mu = x, y (gathered at y)
__global__ void __launch_bounds__(256) k_links_vjp(const double* __restrict__ V, const double* __restrict__ Ub, double* __restrict__ Vb,
                            Geom g) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const int z = (int)(s / g.P);
    const long s2 = s - (long)z * g.P;
    const int x = (int)(s2 % g.nx), y = (int)(s2 / g.nx);
    M3 acc, Vn, Bm, T;
    m3_zero(acc);
    for (int mu = 0; mu < 2; mu++) {
        const long sp = mu == 0 ? sidx(g, x + 1, y, z) : sidx(g, x, y + 1, z);
        const long sm = mu == 0 ? sidx(g, x - 1, y, z) : sidx(g, x, y - 1, z);
        ldm<long>(V, kGPlanes, 0, sp, Vn);
        ldm<long>(Ub, kUPlanes, 18 * mu, s, Bm);
        mul_nd(Vn, Bm, T);  // V(y+mu) Ubar_mu(y)^dag
        m3_axpy(1.0, T, acc);
        ldm<long>(V, kGPlanes, 0, sm, Vn);
        ldm<long>(Ub, kUPlanes, 18 * mu, sm, Bm);
        mul_nn(Vn, Bm, T);  // V(y-mu) Ubar_mu(y-mu)
        m3_axpy(1.0, T, acc);
    }
    stm<long>(Vb, kGPlanes, 0, s, acc);
}

// Reverse of the left-moving Wilson-line scan V(z) = X(z) V(z+1), X(z) = exp(-i A(z) t / sqrt2), in two kernels.
// The total cotangent of V(z) is its own Vbar(z) plus, through V(z-1) = X(z-1) V(z), X(z-1)^dag times that of V(z-1);
// with X(z') ... X(z-1) = V(z') V(z)^dag (V unitary) this is Wbar(z) = V(z) sum_{z' <= z} V(z')^dag Vbar(z'), a running
// sum along z (k_scan_vjp_sum, Wbar in place of Vbar), after which every layer's
// exponential adjoint is independent (k_scan_vjp_site, one thread per site): Xbar = Wbar(z) V(z+1)^dag.
// The sum in runs of z as in k_wilson_scan: each run's total, then the walk from the earlier runs' sum; both
// lines' sums (blockIdx.y) in one launch.  One thread per site took 2 x 225 us at 48 x 48 x 128, the one launch 92.
struct ScanVjp {
    const double* V[2];
    double* Vb[2];
};
__global__ void __launch_bounds__(64 * kScanChunks) k_scan_vjp_sum(ScanVjp A, Geom g) {
    extern __shared__ double ends[];
    const double* const V = blockIdx.y ? A.V[1] : A.V[0];
    double* const Vb = blockIdx.y ? A.Vb[1] : A.Vb[0];
    const int nc = blockDim.x >> 6, c = threadIdx.x >> 6, len = (g.nz + nc - 1) / nc;
    const long s2 = (long)blockIdx.x * 64 + (threadIdx.x & 63);
    const int z0 = min(g.nz, c * len), z1 = s2 < g.P ? min(g.nz, z0 + len) : z0;
    M3 acc, Vz, B, T;
    m3_zero(acc);
    for (int z = z0; z < z1 && c + 1 < nc; z++) {  // the last run's total is not needed
        const long s = s2 + g.P * z;
        ldm<long>(V, kGPlanes, 0, s, Vz);
        ldm<long>(Vb, kGPlanes, 0, s, B);
        mul_dn(Vz, B, T);
        m3_axpy(1.0, T, acc);
    }
    st_end(ends, c, acc);
    __syncthreads();
    m3_zero(acc);
    for (int j = 0; j < c; j++) {
        ld_end(ends, j, T);
        m3_axpy(1.0, T, acc);
    }
    for (int z = z0; z < z1; z++) {
        const long s = s2 + g.P * z;
        ldm<long>(V, kGPlanes, 0, s, Vz);
        ldm<long>(Vb, kGPlanes, 0, s, B);
        mul_dn(Vz, B, T);
        m3_axpy(1.0, T, acc);
        mul_nn(Vz, acc, T);
        stm<long>(Vb, kGPlanes, 0, s, T);
    }
}
// Abar (real, a*S + s) from Wbar
__global__ void __launch_bounds__(256) k_scan_vjp_site(const double* __restrict__ A, const double* __restrict__ V,
                                                       const double* __restrict__ Wb, double* __restrict__ Ab, Geom g) {
    const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const double c = -1.0 / kSqrt2;
    const int z = (int)(s / g.P);
    M3 W, Wn, X, Xb;
    ldm<long>(Wb, kGPlanes, 0, s, W);
    if (z + 1 < g.nz) ldm<long>(V, kGPlanes, 0, s + g.P, Wn);
    else set_unit(Wn);
    double a[8], ab[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int q = 0; q < 8; q++) a[q] = A[(long)q * g.S + s];
    expi(c, a, X);
    mul_nd(W, Wn, Xb);
    dexp_adjoint(c, a, X, Xb, ab);
    for (int q = 0; q < 8; q++) Ab[(long)q * g.S + s] = ab[q];
}

// ------------------------------------------------------------------------------------------------
// Physical-charge (TMD / GBW) nuclei: SC/TMDNUCLEUS/CorrelationFunction.cpp, GBWSampling.cpp, TMDbased.cpp
// and the initial state of SC/SimulationmitPC.cpp:326-370.
// ------------------------------------------------------------------------------------------------
// F = (noise / sqrt(a^3), 0); noise[a + 8 s] (ChargeFluctuation :29-39)
__global__ void k_tmd_noise(double* __restrict__ F, const double* __restrict__ noise, Geom g, double sqrt_acube) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        F[2 * i] = noise[a + 8 * s] / sqrt_acube;
        F[2 * i + 1] = 0.0;
    }
}

// ChargeFluctuation's momentum-space factor (:45-79) on the 3D transform: nf sqrt(GammaK(x, kT^2)) for
// x = |p_z| / (CoMEnergy / sqrt2) <= 1, else 0; |p_z| = sqrt((2 - 2 cos(2 pi n_z / N_z)) / aZInFm^2) / sqrt2;
// GammaK = 4 pi Nc / (Nc^2 - 1) kT^4 / Qs^2 exp(-kT^2 / Qs^2), Qs = Qs0A x^-0.1 (1 - x) / sqrt(ax ay) (:17-22)
__global__ void k_tmd_cf_filter(double* __restrict__ F, Geom g, double ax, double ay, double qs0a, double com_energy,
                                double az_fm) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const int pz = (int)(s / g.P);
    const long s2 = s - (long)pz * g.P;
    const int px = (int)(s2 % g.nx), py = (int)(s2 / g.nx);
    const double pl = (1 / kSqrt2) * sqrt((2.0 - 2.0 * cos(2.0 * kPi * pz / (double)g.nz)) / (az_fm * az_fm));
    const double kT2 = psqr2(g, px, py, ax, ay);
    const double x = pl / (com_energy / kSqrt2);
    const double nf = 1.0 / ((double)g.nx * g.ny * g.nz);
    double f = 0.0;
    if (x <= 1.0) {
        const double Qs = qs0a * pow(x, -0.1) * (1 - x) / sqrt(ax * ay);
        f = sqrt(4.0 * kPi * 3.0 / (3.0 * 3.0 - 1.0) * kT2 * kT2 / (Qs * Qs) * exp(-kT2 / (Qs * Qs)));
    }
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        if (x <= 1.0) {
            F[2 * i] = nf * F[2 * i] * f;
            F[2 * i + 1] = nf * F[2 * i + 1] * f;
        } else {
            F[2 * i] = 0.0;
            F[2 * i + 1] = 0.0;
        }
    }
}

struct TmdCharge {
    const double* pos;  // nucleon positions, 3 per nucleon (fm)
    int A;
    double afm[3];
    double gamma, acube, az;
    int zc;
};

// TmdBasedCollision::SetChargeDensities' charge (TMDbased.cpp:27-57): F = (a^3 sqrt(aZInFm T / a_z) Re F, 0), T the
// nucleus profile (GBWSampling.cpp:110-157) at x = (ix - Nx/2) aXInFm, y = (iy - Ny/2) aYInFm, z = (iz - centre) aZInFm
__global__ void k_tmd_charge(double* __restrict__ F, Geom g, TmdCharge C) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.S) return;
    const int z = (int)(s / g.P);
    const long s2 = s - (long)z * g.P;
    const int ix = (int)(s2 % g.nx), iy = (int)(s2 / g.nx);
    const double x = (ix - g.nx / 2) * C.afm[0], y = (iy - g.ny / 2) * C.afm[1], zf = (z - C.zc) * C.afm[2];
    const double BG = 4.0 * 0.197 * 0.197;
    double T = 0.0;
    for (int n = 0; n < C.A; n++) {
        const double dx = x - C.pos[3 * n], dy = y - C.pos[3 * n + 1], dz = C.gamma * zf - C.pos[3 * n + 2];
        const double d2 = dx * dx + dy * dy + dz * dz;
        T += C.gamma * exp(-0.5 * d2 / BG) / sqrt(2.0 * kPi * BG);
    }
    const double c = C.acube * sqrt(C.afm[2] * T / C.az);
    for (int a = 0; a < 8; a++) {
        const long i = fidx(g, a, s);
        F[2 * i] = c * F[2 * i];
        F[2 * i + 1] = 0.0;
    }
}

bool tmd_valid(const glasma_tmd_params* p) {
    return p && p->qs0a > 0.0 && p->m_eff >= 0.0 && p->com_energy > 0.0 && p->a_fm[0] > 0.0 && p->a_fm[1] > 0.0 &&
           p->a_fm[2] > 0.0 && p->atomic_number > 0;
}

// ChargeFluctuation + TmdBasedCollision::SetWilsonLines for one nucleus: w.rho = filtered charge, w.V
int tmd_wilson_lines(glasma_ctx* ctx, Wk& w, const glasma_tmd_params* p, const double* noise_host,
                     const double* pos_host, bool right) {
    const Geom& g = ctx->g;
    const double* a = ctx->p.a;
    // the noise goes through w.rho (8 S doubles), which the filter step overwrites later
    GL_HIP(ctx, hipMemcpyAsync(w.rho, noise_host, 8 * (size_t)g.S * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    double* pos = nullptr;
    GL_HIP(ctx, hipMalloc(&pos, 3 * (size_t)p->atomic_number * sizeof(double)));
    hipError_t e = hipMemcpyAsync(pos, pos_host, 3 * (size_t)p->atomic_number * sizeof(double), hipMemcpyHostToDevice,
                                  ctx->stream);
    int rc = 0;
    if (e != hipSuccess) rc = hip_fail(ctx, e, "tmd nucleon positions");
    if (!rc) {
        hipLaunchKernelGGL(k_tmd_noise, grid1(g.S), dim3(256), 0, ctx->stream, w.F, w.rho, g, std::sqrt(a[0] * a[1] * a[2]));
        rc = fft_3d(ctx->stream, w.F, g, 8, -1);
        if (!rc) {
            hipLaunchKernelGGL(k_tmd_cf_filter, grid1(g.S), dim3(256), 0, ctx->stream, w.F, g, a[0], a[1], p->qs0a,
                               p->com_energy, p->a_fm[2]);
            rc = fft_3d(ctx->stream, w.F, g, 8, +1);
        }
        if (rc)
            rc = set_error(ctx, rc,
                           std::string("FFT failed (lengths must be 2^a 3^b p <= 2048, prime factors <= 13): ") +
                               fft_last_error());
    }
    if (!rc) {
        TmdCharge C;
        C.pos = pos;
        C.A = p->atomic_number;
        for (int m = 0; m < 3; m++) C.afm[m] = p->a_fm[m];
        C.gamma = p->com_energy * 0.197 / 2.0;
        C.acube = a[0] * a[1] * a[2];
        C.az = a[2];
        C.zc = right ? p->center_r : p->center_l;
        hipLaunchKernelGGL(k_tmd_charge, grid1(g.S), dim3(256), 0, ctx->stream, w.F, g, C);
        rc = wilson_from_charge(ctx, w, std::numeric_limits<double>::infinity(), p->m_eff, right);
    }
    (void)hipStreamSynchronize(ctx->stream);  // the positions buffer is freed below
    (void)hipFree(pos);
    return rc;
}

bool mv_valid(const glasma_mv_params* mv) {
    return mv && mv->sigma_l > 0.0 && mv->sigma_r > 0.0 && mv->lambda > 0.0 && mv->m_eff >= 0.0;
}

}  // namespace

// Left-moving sheet over all z from a given charge density rho (device, real, a*S + s; the density
// SetChargeDensities would produce), keeping the intermediates in tape (device arrays of 8*S doubles
// for rho_s, A0, A1 and tiled 18-plane Wilson lines V0, V1).  Resets the fields and the time first.
int ic_left_from_charge(glasma_ctx* ctx, const glasma_mv_params* mv, const double* rho, IcTape& tape) {
    const Geom& g = ctx->g;
    int rc = reset_fields(ctx);
    if (rc) return rc;
    rc = ensure_fftbuf(ctx, 16 * (size_t)g.S);
    if (rc) return rc;
    double* F = ctx->fftbuf;
    hipStream_t st = ctx->stream;
    double* U = ctx->U[ctx->cur];
    double* J = ctx->J[ctx->cur];
    const double dt = ctx->p.dt;
    hipLaunchKernelGGL(k_load_real, grid1(g.S), dim3(256), 0, st, F, rho, g);
    GL_FFT(ctx, fft_xy(st, F, g, 8, g.nz, -1));
    hipLaunchKernelGGL(k_transverse_filter, grid1(g.S), dim3(256), 0, st, F, g, ctx->p.a[0], ctx->p.a[1], mv->lambda,
                       mv->m_eff, 0);
    GL_FFT(ctx, fft_xy(st, F, g, 8, g.nz, +1));
    hipLaunchKernelGGL(k_take_real, grid1(g.S), dim3(256), 0, st, F, tape.rho_s, g);
    GL_RC(poisson_all(ctx, F));
    hipLaunchKernelGGL(k_copy_real, grid1(8 * g.S), dim3(256), 0, st, tape.A0, F, g);
    GL_RC(wilson_scan(ctx, F, tape.V0, 0));
    hipLaunchKernelGGL(k_sheet_links, grid1(g.S), dim3(256), 0, st, tape.V0, ctx->UOld, g, 0, g.nz - 1);
    hipLaunchKernelGGL(k_load_real, grid1(g.S), dim3(256), 0, st, F, tape.rho_s, g);
    GL_FFT(ctx, fft_z(st, F, g, 8, -1));
    hipLaunchKernelGGL(k_evolve_phase, grid1(g.S), dim3(256), 0, st, F, g, ctx->p.a[2], dt, 0);
    GL_FFT(ctx, fft_z(st, F, g, 8, +1));
    hipLaunchKernelGGL(k_take_real, grid1(g.S), dim3(256), 0, st, F, (double*)nullptr, g);
    GL_RC(poisson_all(ctx, F));
    hipLaunchKernelGGL(k_copy_real, grid1(8 * g.S), dim3(256), 0, st, tape.A1, F, g);
    GL_RC(wilson_scan(ctx, F, tape.V1, 0));
    hipLaunchKernelGGL(k_sheet_links, grid1(g.S), dim3(256), 0, st, tape.V1, U, g, 0, g.nz - 1);
    const double acube = ctx->p.a[0] * ctx->p.a[1] * ctx->p.a[2];
    const double coff0 = -dt * ctx->p.a[0] * ctx->p.a[0] / acube;
    const double coff1 = -dt * ctx->p.a[1] * ctx->p.a[1] / acube;
    hipLaunchKernelGGL(k_sheet_efield, efield_grid(g.S), dim3(256), 0, st, U, ctx->UOld, ctx->E, g, 0, g.nz - 1, coff0, coff1);
    SheetSides A;
    A.n = 1;
    A.s[0] = sheet_side(false, 0, g.nz - 1, JPS, JP);
    return sheet_currents(ctx, U, ctx->E, J, A);
}

// Reverse-mode derivative of ic_left_from_charge.  In: cotangents of the sheet's U (Ub, tiled 54 planes;
// modified), E (Eb, tiled 24; modified) and J (Jb, tiled 32: J+ and J+stat used), the fields and tape of
// the same call.  Out: rho_bar (device, real, a*S + s).  work: 54*Sp + 2*18*Sp + 4*8*S doubles.
int ic_left_vjp(glasma_ctx* ctx, const glasma_mv_params* mv, const IcTape& tape, double* Ub, double* Eb,
                const double* Jb, double* rho_bar, double* work) {
    const Geom& g = ctx->g;
    const long Sp = pad_sites(g.S);
    hipStream_t st = ctx->stream;
    int rc = ensure_fftbuf(ctx, 16 * (size_t)g.S);
    if (rc) return rc;
    double* F = ctx->fftbuf;
    double* UOb = work;
    double* V0b = UOb + 54 * Sp;
    double* V1b = V0b + 18 * Sp;
    double* jsb = V1b + 18 * Sp;
    double* A0b = jsb + 8 * g.S;
    double* A1b = A0b + 8 * g.S;
    double* tmp = A1b + 8 * g.S;
    const double* U = ctx->U[ctx->cur];
    const double dt = ctx->p.dt;
    // J+ = jinv(J+stat): J+stat cotangent += jinv^T(J+ cotangent)
    hipLaunchKernelGGL(k_load_planes, grid1(g.S), dim3(256), 0, st, F, Jb, g, kJPlanes, 8 * JP);
    GL_FFT(ctx, fft_z(st, F, g, 8, -1));
    hipLaunchKernelGGL(k_jinv, grid1(g.S), dim3(256), 0, st, F, g, ctx->p.a[2], dt, 0, 1);
    GL_FFT(ctx, fft_z(st, F, g, 8, +1));
    hipLaunchKernelGGL(k_copy_real, grid1(8 * g.S), dim3(256), 0, st, tmp, F, g);
    hipLaunchKernelGGL(k_load_planes, grid1(g.S), dim3(256), 0, st, F, Jb, g, kJPlanes, 8 * JPS);
    hipLaunchKernelGGL(k_axpy_real, grid1(8 * g.S), dim3(256), 0, st, jsb, tmp, F, 1.0, g);
    // J+stat from E and U
    hipLaunchKernelGGL(k_ic_jstat_vjp, grid1(g.S), dim3(256), 0, st, U, ctx->E, jsb, Ub, Eb, g);
    // E = ilog(U UOld^dag)
    const double acube = ctx->p.a[0] * ctx->p.a[1] * ctx->p.a[2];
    const double coff0 = -dt * ctx->p.a[0] * ctx->p.a[0] / acube;
    const double coff1 = -dt * ctx->p.a[1] * ctx->p.a[1] / acube;
    hipLaunchKernelGGL(k_zero, grid1(54 * Sp), dim3(256), 0, st, UOb, 54 * Sp);
    hipLaunchKernelGGL(k_ic_ilog_vjp, grid1(g.S), dim3(256), 0, st, U, ctx->UOld, ctx->E, Eb, Ub, UOb, g, coff0, coff1);
    // links -> Wilson lines -> Poisson solutions
    hipLaunchKernelGGL(k_links_vjp, grid1(g.S), dim3(256), 0, st, tape.V1, Ub, V1b, g);
    hipLaunchKernelGGL(k_links_vjp, grid1(g.S), dim3(256), 0, st, tape.V0, UOb, V0b, g);
    const int nc = scan_chunks(g);
    GL_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void*>(&k_scan_vjp_sum),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)scan_lds(kScanChunks)));
    hipLaunchKernelGGL(k_scan_vjp_sum, dim3((unsigned)((g.P + 63) / 64), 2), dim3(64 * nc), scan_lds(nc), st,
                       ScanVjp{{tape.V1, tape.V0}, {V1b, V0b}}, g);
    hipLaunchKernelGGL(k_scan_vjp_site, grid1(g.S), dim3(256), 0, st, tape.A1, tape.V1, V1b, A1b, g);
    hipLaunchKernelGGL(k_scan_vjp_site, grid1(g.S), dim3(256), 0, st, tape.A0, tape.V0, V0b, A0b, g);
    // rho_ev cotangent = poisson(A1bar); rho_s cotangent = evolve_R(that) + poisson(A0bar)
    hipLaunchKernelGGL(k_load_real, grid1(g.S), dim3(256), 0, st, F, A1b, g);
    GL_RC(poisson_all(ctx, F));
    hipLaunchKernelGGL(k_take_real, grid1(g.S), dim3(256), 0, st, F, (double*)nullptr, g);
    GL_FFT(ctx, fft_z(st, F, g, 8, -1));
    hipLaunchKernelGGL(k_evolve_phase, grid1(g.S), dim3(256), 0, st, F, g, ctx->p.a[2], dt, 1);
    GL_FFT(ctx, fft_z(st, F, g, 8, +1));
    hipLaunchKernelGGL(k_copy_real, grid1(8 * g.S), dim3(256), 0, st, tmp, F, g);
    hipLaunchKernelGGL(k_load_real, grid1(g.S), dim3(256), 0, st, F, A0b, g);
    GL_RC(poisson_all(ctx, F));
    hipLaunchKernelGGL(k_axpy_real, grid1(8 * g.S), dim3(256), 0, st, tmp, tmp, F, 1.0, g);
    // rho cotangent = smooth(rho_s cotangent)
    hipLaunchKernelGGL(k_load_real, grid1(g.S), dim3(256), 0, st, F, tmp, g);
    GL_FFT(ctx, fft_xy(st, F, g, 8, g.nz, -1));
    hipLaunchKernelGGL(k_transverse_filter, grid1(g.S), dim3(256), 0, st, F, g, ctx->p.a[0], ctx->p.a[1], mv->lambda,
                       mv->m_eff, 0);
    GL_FFT(ctx, fft_xy(st, F, g, 8, g.nz, +1));
    hipLaunchKernelGGL(k_copy_real, grid1(8 * g.S), dim3(256), 0, st, rho_bar, F, g);
    GL_HIP(ctx, hipGetLastError());
    return 0;
}

}  // namespace glasma

using namespace glasma;

namespace glasma {
namespace {
// The part of reset_fields a sheet initial state needs.  The sheets write the current links, UOld and E at every
// site (the collision's two sheets cover [0, (Nz-2)/2] and [Nz/2, Nz-1], a single nucleus all of z), and whole planes
// of the current J (k_sheet_jstat, k_sheet_jinv); the planes of the nucleus a single-nucleus driver leaves out must be
// zero.  The other buffers of the ping-pong pairs are written by the first step before anything reads them.
int reset_for_sheets(glasma_ctx* ctx, int driver) {
    ctx->cur = 0;
    ctx->t = 0.0;
    ctx->tsteps = 0;
    if (driver != 0)
        GL_HIP(ctx, hipMemsetAsync(ctx->J[0], 0, (size_t)kJPlanes * pad_sites(ctx->g.S) * sizeof(double), ctx->stream));
    return 0;
}
}  // namespace
}  // namespace glasma

extern "C" int glasma_mv_initial_state(glasma_ctx* ctx, int driver, const glasma_mv_params* mv, const double* xi_l,
                                       const double* xi_r) {
    if (!ctx) return GLASMA_ERR_ARG;
    if (!mv_valid(mv)) return set_error(ctx, GLASMA_ERR_ARG, "invalid MV parameters");
    if (driver < 0 || driver > 2) return set_error(ctx, GLASMA_ERR_ARG, "driver must be 0, 1 or 2");
    if ((driver != 2 && !xi_l) || (driver != 1 && !xi_r)) return set_error(ctx, GLASMA_ERR_ARG, "missing charges");
    int rc = reset_for_sheets(ctx, driver);
    if (rc) return rc;
    const int nz = ctx->g.nz;
    // collision: left sheet on [0, (Nz-2)/2] (SC/Simulation.cpp:359), right on [Nz/2, Nz-1]; single nucleus: all z
    SheetSides sides;
    const double* xi[2] = {xi_l, xi_r};
    sides.n = 0;
    if (driver != 2) sides.s[sides.n++] = sheet_side(false, 0, driver == 0 ? (nz - 2) / 2 : nz - 1, JPS, JP);
    if (driver != 1) {
        xi[sides.n] = xi_r;
        sides.s[sides.n++] = sheet_side(true, driver == 0 ? nz / 2 : 0, nz - 1, JMS, JM);
    }
    Wk w;
    if (mv->m_eff > 0.0) {
        if (sides.n == 2 && nz == 1) {  // the two ranges overlap: the right sheet after the left
            SheetSides one;
            one.n = 1;
            for (int k = 0; k < 2 && rc == 0; k++) {
                one.s[0] = sides.s[k];
                rc = mv_sheets(ctx, mv, one, xi + k);
            }
        } else {
            rc = mv_sheets(ctx, mv, sides, xi);
        }
    } else {
        rc = alloc_work(ctx, w);
        for (int k = 0; k < sides.n && rc == 0; k++) {
            const SheetSide& sd = sides.s[k];
            rc = set_wilson_lines(ctx, w, mv, xi[k], sd.right != 0);
            if (rc == 0) rc = single_sheet(ctx, w, sd.right != 0, sd.zlo, sd.zhi, sd.wstat, sd.wj);
        }
    }
    if (rc == 0) {
        hipError_t e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) rc = hip_fail(ctx, e, "mv_initial_state");
    }
    free_work(w);
    return rc;
}

extern "C" int glasma_tmd_initial_state(glasma_ctx* ctx, int driver, const glasma_tmd_params* p, const double* noise_l,
                                        const double* noise_r, const double* nucleons_l, const double* nucleons_r) {
    if (!ctx) return GLASMA_ERR_ARG;
    if (!tmd_valid(p)) return set_error(ctx, GLASMA_ERR_ARG, "invalid physical-charge parameters");
    if (driver < 0 || driver > 2) return set_error(ctx, GLASMA_ERR_ARG, "driver must be 0, 1 or 2");
    if ((driver != 2 && (!noise_l || !nucleons_l)) || (driver != 1 && (!noise_r || !nucleons_r)))
        return set_error(ctx, GLASMA_ERR_ARG, "missing noise or nucleon positions");
    int rc = reset_for_sheets(ctx, driver);
    if (rc) return rc;
    const int nz = ctx->g.nz;
    Wk w;
    rc = alloc_work(ctx, w);
    if (rc == 0 && driver != 2) {
        const int zhi = driver == 0 ? (nz - 2) / 2 : nz - 1;
        rc = tmd_wilson_lines(ctx, w, p, noise_l, nucleons_l, false);
        if (rc == 0) rc = single_sheet(ctx, w, false, 0, zhi, JPS, JP);
    }
    if (rc == 0 && driver != 1) {
        const int zlo = driver == 0 ? nz / 2 : 0;
        rc = tmd_wilson_lines(ctx, w, p, noise_r, nucleons_r, true);
        if (rc == 0) rc = single_sheet(ctx, w, true, zlo, nz - 1, JMS, JM);
    }
    if (rc == 0) {
        hipError_t e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) rc = hip_fail(ctx, e, "tmd_initial_state");
    }
    free_work(w);
    return rc;
}

extern "C" int glasma_set_wilson_lines(glasma_ctx* ctx, char dir, const glasma_mv_params* mv, const double* xi,
                                       double* V_out, double* rho_out) {
    if (!ctx) return GLASMA_ERR_ARG;
    if (!mv_valid(mv) || !xi || (dir != 'L' && dir != 'R'))
        return set_error(ctx, GLASMA_ERR_ARG, "invalid arguments to glasma_set_wilson_lines");
    Wk w;
    int rc = alloc_work(ctx, w);
    if (rc == 0) rc = set_wilson_lines(ctx, w, mv, xi, dir == 'R');
    if (rc == 0 && V_out) rc = download_aos(ctx, w.V, V_out, kGPlanes);
    if (rc == 0 && rho_out) {
        const Geom& g = ctx->g;
        double* tmp = nullptr;
        hipError_t e = hipMalloc(&tmp, 8 * (size_t)g.S * sizeof(double));
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_rho_to_aos, grid1(8 * g.S), dim3(256), 0, ctx->stream, w.rho, tmp, g);
            e = hipGetLastError();
            if (e == hipSuccess)
                e = hipMemcpyAsync(rho_out + 8 * g.P, tmp, 8 * (size_t)g.S * sizeof(double), hipMemcpyDeviceToHost,
                                   ctx->stream);
            if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
            (void)hipFree(tmp);
        }
        if (e != hipSuccess) rc = hip_fail(ctx, e, "set_wilson_lines rho");
        else host_sync_ghosts(ctx, rho_out, 8);
    }
    free_work(w);
    return rc;
}
