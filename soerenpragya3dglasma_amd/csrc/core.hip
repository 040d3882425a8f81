// libglasma core: context lifetime, field transfer between the reference AoS layout and the device
// SoA layout, the time loop entry points and the observable reductions.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <vector>

#include "internal.h"

namespace glasma {

int launch_step(glasma_ctx* ctx, bool write_old);

int set_error(glasma_ctx* ctx, int code, const std::string& msg) {
    if (ctx) ctx->err = msg;
    return code;
}
int hip_code(hipError_t e) {
    (void)hipGetLastError();
    return e == hipErrorOutOfMemory ? GLASMA_ERR_NOMEM : GLASMA_ERR_HIP;
}
int hip_fail(glasma_ctx* ctx, hipError_t e, const char* what) {
    std::string m = std::string(what) + ": " + hipGetErrorString(e);
    return set_error(ctx, hip_code(e), m);
}
int ensure_red(glasma_ctx* ctx, size_t doubles) {
    if (ctx->red_cap >= doubles) return 0;
    if (ctx->red) (void)hipFree(ctx->red);
    ctx->red = nullptr;
    ctx->red_cap = 0;
    GL_HIP(ctx, hipMalloc(&ctx->red, doubles * sizeof(double)));
    ctx->red_cap = doubles;
    return 0;
}
int ensure_fftbuf(glasma_ctx* ctx, size_t doubles) {
    if (ctx->fftbuf_cap >= doubles) return 0;
    if (ctx->fftbuf) (void)hipFree(ctx->fftbuf);
    ctx->fftbuf = nullptr;
    ctx->fftbuf_cap = 0;
    GL_HIP(ctx, hipMalloc(&ctx->fftbuf, doubles * sizeof(double)));
    ctx->fftbuf_cap = doubles;
    return 0;
}

static int upload_j(glasma_ctx* ctx, const double* h, double* J, int w) { return upload_aos(ctx, h, J, 8, kJPlanes, 8 * w); }
static int download_j(glasma_ctx* ctx, const double* J, double* h, int w) {
    return download_aos(ctx, J, h, 8, kJPlanes, 8 * w);
}

// identity links / zero fields
// identity matrices in all nmat matrix slots of a field with 18*nmat planes
__global__ void k_set_identity(double* __restrict__ U, long S, int nmat) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S) return;
    for (int m = 0; m < nmat; m++)
        for (int e = 0; e < 18; e++)
            U[lidx<long>(18 * nmat, 18 * m + e, s)] = (e == 0 || e == 8 || e == 16) ? 1.0 : 0.0;
}

// counter-based uniform in (0,1): splitmix64 finaliser of (seed, index)
__device__ __forceinline__ double hash_uniform(unsigned long long seed, unsigned long long i) {
    unsigned long long z = seed * 0x9E3779B97F4A7C15ull + i * 0xD1B54A32D192ED03ull + 0x632BE59BD9B4E019ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return ((double)(z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}
// uniform in [-1, 1) per component: links exp(i s_U alpha t) with alpha_a uniform, E and J uniform
__global__ void __launch_bounds__(256) k_fill_random(double* __restrict__ U, double* __restrict__ E, double* __restrict__ J, long S,
                              unsigned long long seed, double su, double se, double sj) {
    long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= S) return;
    unsigned long long base = (unsigned long long)s * 64ull;
    for (int mu = 0; mu < 3; mu++) {
        double al[8];
        for (int a = 0; a < 8; a++) al[a] = 2.0 * hash_uniform(seed, base + mu * 8 + a) - 1.0;
        M3 X;
        expi(su, al, X);
        stm<long>(U, kUPlanes, 18 * mu, s, X);
        for (int a = 0; a < 8; a++)
            E[lidx<long>(kEPlanes, mu * 8 + a, s)] = se * (2.0 * hash_uniform(seed ^ 0x5555ull, base + mu * 8 + a) - 1.0);
    }
    for (int w = 0; w < 4; w++)
        for (int a = 0; a < 8; a++)
            J[lidx<long>(kJPlanes, w * 8 + a, s)] = sj * (2.0 * hash_uniform(seed ^ 0xAAAAull, base + w * 8 + a) - 1.0);
}

int reset_fields(glasma_ctx* ctx) {
    const long S = ctx->g.S;
    dim3 grid((unsigned)((S + 255) / 256));
    hipLaunchKernelGGL(k_set_identity, grid, dim3(256), 0, ctx->stream, ctx->U[0], S, 3);
    hipLaunchKernelGGL(k_set_identity, grid, dim3(256), 0, ctx->stream, ctx->U[1], S, 3);
    hipLaunchKernelGGL(k_set_identity, grid, dim3(256), 0, ctx->stream, ctx->UOld, S, 3);
    const long Sp = pad_sites(S);
    GL_HIP(ctx, hipMemsetAsync(ctx->E, 0, (size_t)kEPlanes * Sp * sizeof(double), ctx->stream));
    GL_HIP(ctx, hipMemsetAsync(ctx->J[0], 0, (size_t)kJPlanes * Sp * sizeof(double), ctx->stream));
    GL_HIP(ctx, hipMemsetAsync(ctx->J[1], 0, (size_t)kJPlanes * Sp * sizeof(double), ctx->stream));
    GL_HIP(ctx, hipStreamSynchronize(ctx->stream));
    ctx->cur = 0;
    ctx->t = 0.0;
    ctx->tsteps = 0;
    return 0;
}

// ------------------------------------------------------------------------------------------------
// observables
// ------------------------------------------------------------------------------------------------
// One block of 256 threads per (chunk of a z plane); partial sums of K quantities per block are
// written to red[(z*bpp + b)*K + k] and summed afterwards in a fixed order: results do not depend on
// scheduling and are reproducible bit for bit.
template <int K>
__device__ __forceinline__ void block_store(double (&v)[K], double* out) {
    __shared__ double sh[4][K];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = wave_sum(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < K; k++) sh[wid][k] = v[k];
    __syncthreads();
    if (threadIdx.x < K) {
        const int k = threadIdx.x;
        out[k] = ((sh[0][k] + sh[1][k]) + sh[2][k]) + sh[3][k];
    }
}
template <int K>
__device__ __forceinline__ void block_store_max(double (&v)[K], double* out) {
    __shared__ double shm[4][K];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = wave_max(v[k]);
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < K; k++) shm[wid][k] = v[k];
    __syncthreads();
    if (threadIdx.x < K) {
        const int k = threadIdx.x;
        out[k] = fmax(fmax(shm[0][k], shm[1][k]), fmax(shm[2][k], shm[3][k]));
    }
}

// Which 256-site chunk of which plane a block of a record kernel takes (block b runs on XCD b % 8, each XCD with its own
// L2).  band > 0: XCD k takes the bands k, k + 8, ... of `band` consecutive chunks of a plane and walks each through all
// layers, so that the layers of a band in flight at once share their y and z neighbours in L2; band = 0: XCD k takes the
// k-th eighth of the chunks, layer by layer.  With chunks dealt to the XCDs in turn the energy-momentum kernel fetched
// 4.4 times its compulsory bytes at 256 x 256 x 128.
struct ObsOrder {
    int bpp, nz, band;
    unsigned n, per;  // blocks, blocks per XCD (far below 2^32 on any device memory)
};
static ObsOrder obs_order(int bpp, int nz) {
    const unsigned n = (unsigned)bpp * (unsigned)nz;
    ObsOrder o = {bpp, nz, 0, n, (n + kXcds - 1) / kXcds};
    for (int b = 1; b <= 16; b++)
        if (bpp % b == 0 && bpp / b % kXcds == 0) o.band = b;
    return o;
}
__device__ __forceinline__ bool obs_block(const ObsOrder& o, int& chunk, int& z) {
    const unsigned k = blockIdx.x % kXcds, i = blockIdx.x / kXcds;
    if (o.band) {
        const unsigned per = (unsigned)o.band * o.nz, m = i / per, r = i - m * per;
        z = (int)(r / o.band);
        chunk = (int)((m * kXcds + k) * o.band + r % o.band);
        return true;
    }
    const unsigned b = k * o.per + i;
    z = (int)(b / o.bpp);
    chunk = (int)(b % o.bpp);
    return b < o.n;
}

struct ObsArgs {
    const double* __restrict__ U;
    const double* __restrict__ UOld;
    const double* __restrict__ E;
    const double* __restrict__ J;
    double* __restrict__ red;
    Geom g;
    int bpp;  // blocks per plane
    ObsOrder ord;
    double a[3];
};

// the block's place for its partial sums (null: no chunk) and the thread's site (false: none)
template <int K>
__device__ __forceinline__ double* part_of(const ObsArgs& A, int& chunk, int& z) {
    return obs_block(A.ord, chunk, z) ? A.red + ((long)z * A.bpp + chunk) * K : nullptr;
}
__device__ __forceinline__ bool site_of(const ObsArgs& A, int chunk, int& x, int& y, int z, long& s) {
    const unsigned i = chunk * 256u + threadIdx.x;  // P sites of a plane: far below 2^32 on any device memory
    if (i >= A.g.P) return false;
    x = (int)(i % (unsigned)A.g.nx);
    y = (int)(i / (unsigned)A.g.nx);
    s = i + A.g.P * z;
    return true;
}

// B_k^2 = 4 Re tr(1 - P_k) of the plaquettes P_0 = P_yz, P_1 = P_zx, P_2 = P_xy rooted at a site, each as Re tr(A B^dag)
// of its two corner products A = U_m(x) U_n(x+m) and B = U_n(x) U_m(x+n): two matrix products a plaquette, the third is
// only needed on its diagonal (tr_nd).  What bounds this is how many loads are in flight: the nine links are all read
// before the first product, at one wavefront per SIMD (286 registers for k_bulk).  Pairs of links at three wavefronts
// per SIMD took 1.59 ms for the bulk sums at 128 x 128 x 384, three whole plaquettes of four links 0.97, this 0.93
// (752 B per site, 5.1 TB/s).
__device__ __forceinline__ void site_b2(const double* __restrict__ U, const Geom& g, int x, int y, int z, long s,
                                        double* b) {
    const long sxp = sidx(g, x + 1, y, z), syp = sidx(g, x, y + 1, z), szp = sidx(g, x, y, zup(g, z));
    M3 X, Y, Z, Yx, Zx, Xy, Zy, Xz, Yz, A, B;
    ldm<long>(U, kUPlanes, 0, s, X);
    ldm<long>(U, kUPlanes, 18, s, Y);
    ldm<long>(U, kUPlanes, 18, sxp, Yx);
    ldm<long>(U, kUPlanes, 0, syp, Xy);
    ldm<long>(U, kUPlanes, 36, s, Z);
    ldm<long>(U, kUPlanes, 36, syp, Zy);
    ldm<long>(U, kUPlanes, 18, szp, Yz);
    ldm<long>(U, kUPlanes, 0, szp, Xz);
    ldm<long>(U, kUPlanes, 36, sxp, Zx);
    mul_nn(X, Yx, A);
    mul_nn(Y, Xy, B);
    b[2] = 4.0 * (3.0 - tr_nd(A, B));
    mul_nn(Y, Zy, A);
    mul_nn(Z, Yz, B);
    b[0] = 4.0 * (3.0 - tr_nd(A, B));
    mul_nn(Z, Xz, A);
    mul_nn(X, Zx, B);
    b[1] = 4.0 * (3.0 - tr_nd(A, B));
}
// E_mu^2 of a site
__device__ __forceinline__ double site_e2(const double* __restrict__ E, int mu, long s) {
    double e[8], v = 0.0;
    ldv<long>(E, kEPlanes, 8 * mu, s, e);
#pragma unroll
    for (int a = 0; a < 8; a++) v += e[a] * e[a];
    return v;
}
// Observables::Bulk (SC/OBSERVABLES/BulkObservables.cpp:65-169): K = 9 (E^2[3], B^2[3], E.J[3])
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) k_bulk(ObsArgs A) {
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    int chunk, x, y, z;
    long s;
    double* const out = part_of<9>(A, chunk, z);
    if (!out) return;
    if (site_of(A, chunk, x, y, z, s)) {
        site_b2(A.U, A.g, x, y, z, s, v + 3);
        v[0] = site_e2(A.E, 0, s);
        v[1] = site_e2(A.E, 1, s);
        double e[8], jp[8], jm[8];
        ldv<long>(A.E, kEPlanes, 16, s, e);
        ldv<long>(A.J, kJPlanes, 8 * JP, s, jp);
        ldv<long>(A.J, kJPlanes, 8 * JM, s, jm);
#pragma unroll
        for (int a = 0; a < 8; a++) {
            v[2] += e[a] * e[a];
            v[8] += e[a] * (jp[a] - jm[a]) / kSqrt2;
        }
    }
    block_store<9>(v, out);
}

// COMPUTE_GAUSS_VIOLATION (SC/CALC/GaussViolation.cpp:13-23): K = 2 sums (sum G^2) + 1 max (|G^a|)
__global__ void __launch_bounds__(256) k_gauss(ObsArgs A) {
    double v[1] = {0.0};
    double m[1] = {0.0};
    int chunk, x, y, z;
    long s;
    double* const out = part_of<2>(A, chunk, z);
    if (!out) return;
    if (site_of(A, chunk, x, y, z, s)) {
        const Geom& g = A.g;
        const long sxm = sidx(g, x - 1, y, z), sym = sidx(g, x, y - 1, z), szm = sidx(g, x, y, zdn(g, z));
        const double norm = 1.0 / (A.a[0] * A.a[1] * A.a[2]);
        M3 V;
        double e[8], xd[8], yd[8], zd[8];
        ldm<long>(A.U, kUPlanes, 0, sxm, V);
        ldv<long>(A.E, kEPlanes, 0, sxm, e);
        inv_adj_mul(V, e, xd);
        ldm<long>(A.U, kUPlanes, 18, sym, V);
        ldv<long>(A.E, kEPlanes, 8, sym, e);
        inv_adj_mul(V, e, yd);
        ldm<long>(A.U, kUPlanes, 36, szm, V);
        ldv<long>(A.E, kEPlanes, 16, szm, e);
        inv_adj_mul(V, e, zd);
        double ex[8], ey[8], ez[8], jp[8], jm[8];
        ldv<long>(A.E, kEPlanes, 0, s, ex);
        ldv<long>(A.E, kEPlanes, 8, s, ey);
        ldv<long>(A.E, kEPlanes, 16, s, ez);
        ldv<long>(A.J, kJPlanes, 8 * JPS, s, jp);
        ldv<long>(A.J, kJPlanes, 8 * JMS, s, jm);
#pragma unroll
        for (int a = 0; a < 8; a++) {
            const double G = norm * ((ex[a] - xd[a]) + (ey[a] - yd[a]) + (ez[a] - zd[a]) - (jp[a] + jm[a]) / kSqrt2);
            v[0] += G * G;
            m[0] = fmax(m[0], fabs(G));
        }
    }
    block_store<1>(v, out);
    block_store_max<1>(m, out + 1);
}

// Unitarity (SC/OBSERVABLES/UnitarityViolation.cpp:13-51): sum of squares and max
__global__ void __launch_bounds__(256) k_unitarity(ObsArgs A) {
    double v[1] = {0.0}, m[1] = {0.0};
    int chunk, x, y, z;
    long s;
    double* const out = part_of<2>(A, chunk, z);
    if (!out) return;
    if (site_of(A, chunk, x, y, z, s)) {
        for (int mu = 0; mu < 3; mu++) {
            M3 V;
            ldm<long>(A.U, kUPlanes, 18 * mu, s, V);
            const double n = unitarity_norm(V);
            v[0] += n * n;
            m[0] = fmax(m[0], n);
        }
    }
    block_store<1>(v, out);
    block_store_max<1>(m, out + 1);
}

// Re tr(A B)
__device__ __forceinline__ double tr_nn(const M3& A, const M3& B) {
    double r = 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            r = fma(A.re[mi(i, j)], B.re[mi(j, i)], r);
            r = fma(-A.im[mi(i, j)], B.im[mi(j, i)], r);
        }
    return r;
}

// The clover of the plane (m, n) at s: b = 2 Re tr(i t^a C) and b2 = 4 Re tr(1 - C) of the mean C of its four leaves
// (SC/SUNc/AdvancedOperations.cpp:35-40).  With the spokes a = U_m(x), b = U_n(x), c = U_m(x-m), d = U_n(x-n) and the
// outer corners A1 = U_n(x+m) U_m^dag(x+n), A2 = U_m^dag(x-m+n) U_n^dag(x-m), A3 = U_m(x-n) U_n(x-n+m),
// A4 = U_n^dag(x-m-n) U_m(x-m-n) the leaves are a A1 b^dag, b A2 c, d^dag A3 a^dag and c^dag A4 d.  Re tr(i t^a X^dag) =
// -Re tr(i t^a X), so the projection is that of a (A1 b^dag - A3^dag d) + (b A2 - d^dag A4^dag) c, and the traces add with
// the other signs: ten products and twelve links (four leaves on their own: twelve and sixteen).
__device__ __forceinline__ void clover(const double* __restrict__ W, const Geom& g, int m, int n, int x, int y, int z,
                                       double* b, double& b2) {
    auto at = [&](int sm, int sn) { return nbr<long>(g, x, y, z, m, sm, n, sn); };
    M3 Y1, Z1, Y, T;
    {
        M3 G[3], H[2], A;
        ld_group<long, 3>(W, kUPlanes, 18 * n, {at(0, 0), at(1, 0), at(-1, 0)}, G);
        ld_group<long, 2>(W, kUPlanes, 18 * m, {at(0, 1), at(-1, 1)}, H);
        mul_nd(G[1], H[0], A);
        mul_nd(A, G[0], Y1);
        mul_dd(H[1], G[2], A);
        mul_nn(G[0], A, Z1);
    }
    M3 Y2, Z2;
    {
        M3 G[3], H[2], A;
        ld_group<long, 3>(W, kUPlanes, 18 * n, {at(0, -1), at(1, -1), at(-1, -1)}, G);
        ld_group<long, 2>(W, kUPlanes, 18 * m, {at(0, -1), at(-1, -1)}, H);
        mul_nn(H[0], G[1], A);
        mul_dn(A, G[0], Y2);
        mul_dn(G[2], H[1], A);
        mul_dd(G[0], A, Z2);
    }
    M3 S[2];
    ld_group<long, 2>(W, kUPlanes, 18 * m, {at(0, 0), at(-1, 0)}, S);
    double t = tr_nn(S[0], Y1) + tr_nn(S[0], Y2) + tr_nn(Z1, S[1]) + tr_nn(Z2, S[1]);
#pragma unroll
    for (int k = 0; k < 9; k++) {
        Y.re[k] = Y1.re[k] - Y2.re[k];
        Y.im[k] = Y1.im[k] - Y2.im[k];
        Z1.re[k] -= Z2.re[k];
        Z1.im[k] -= Z2.im[k];
    }
    double f[8];
    retr_igen_prod(S[0], Y, b);
    retr_igen_prod(Z1, S[1], f);
#pragma unroll
    for (int a = 0; a < 8; a++) b[a] = 0.5 * (b[a] + f[a]);
    b2 = 4.0 * (3.0 - 0.25 * t);
}

// EnergyMomentumTensor::CreateMap (SC/OBSERVABLES/EnergyMomentumTensor.cpp:92-170) with
// COMPUTE_AVG_FIELD_STRENGTH (SC/CALC/AvgFieldStrength.cpp:68-145): clover B on UOld, E averaged over
// x and x - mu (colour vectors parallel transported with the current U).  K = 10.
// What bounds it is the links' way from L2: sixteen links a clover in four separate leaves took 16.5 ms at
// 256 x 256 x 512.
__global__ void __launch_bounds__(256) k_emt(ObsArgs A) {
    double v[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    int chunk, x, y, z;
    long s;
    double* const out = part_of<10>(A, chunk, z);
    if (!out) return;
    if (site_of(A, chunk, x, y, z, s)) {
        const Geom& g = A.g;
        const long s0 = s;
        const long sxm = sidx(g, x - 1, y, z), sym = sidx(g, x, y - 1, z), szm = sidx(g, x, y, zdn(g, z));
        double B0[8], B1[8], B2[8], B0S, B1S, B2S;
        clover(A.UOld, g, 0, 1, x, y, z, B2, B2S);
        clover(A.UOld, g, 0, 2, x, y, z, B1, B1S);  // the xz plane: its leaves are the zx plane's, reversed
#pragma unroll
        for (int a = 0; a < 8; a++) B1[a] = -B1[a];
        clover(A.UOld, g, 1, 2, x, y, z, B0, B0S);
        double E0[8], E1[8], E2[8], E0S, E1S, E2S;
        auto avg = [&](int mu, long sm, double* Em, double& es) {
            M3 V;
            double e[8], ed[8];
            ldm<long>(A.U, kUPlanes, 18 * mu, sm, V);
            ldv<long>(A.E, kEPlanes, 8 * mu, sm, e);
            ldv<long>(A.E, kEPlanes, 8 * mu, s0, Em);
            inv_adj_mul(V, e, ed);
            es = 0.0;
#pragma unroll
            for (int a = 0; a < 8; a++) {
                es += 0.5 * (Em[a] * Em[a] + e[a] * e[a]);
                Em[a] = 0.5 * (Em[a] + ed[a]);
            }
        };
        avg(0, sxm, E0, E0S);
        avg(1, sym, E1, E1S);
        avg(2, szm, E2, E2S);
        double q0 = A.a[0] / (A.a[0] * A.a[1] * A.a[2]), q1 = A.a[1] / (A.a[0] * A.a[1] * A.a[2]),
               q2 = A.a[2] / (A.a[0] * A.a[1] * A.a[2]);
        const double inv = 1.0 / (double)g.P;
        auto dot = [](const double* p, const double* r) {
            double acc = 0.0;
            for (int a = 0; a < 8; a++) acc += p[a] * r[a];
            return acc;
        };
        const double Q0 = q0 * q0, Q1 = q1 * q1, Q2 = q2 * q2;
        v[0] = (0.5 * (Q0 * E0S + Q1 * E1S + Q2 * E2S + Q0 * B0S + Q1 * B1S + Q2 * B2S)) * inv;
        v[1] = (0.5 * ((Q1 * E1S + Q2 * E2S + Q1 * B1S + Q2 * B2S) - (Q0 * E0S + Q0 * B0S))) * inv;
        v[2] = (0.5 * ((Q0 * E0S + Q2 * E2S + Q0 * B0S + Q2 * B2S) - (Q1 * E1S + Q1 * B1S))) * inv;
        v[3] = (0.5 * ((Q0 * E0S + Q1 * E1S + Q0 * B0S + Q1 * B1S) - (Q2 * E2S + Q2 * B2S))) * inv;
        v[4] = (q1 * q2 * dot(E1, B2) - q2 * q1 * dot(E2, B1)) * inv;
        v[5] = (q2 * q0 * dot(E2, B0) - q0 * q2 * dot(E0, B2)) * inv;
        v[6] = (q0 * q1 * dot(E0, B1) - q1 * q0 * dot(E1, B0)) * inv;
        v[7] = (q0 * q1 * dot(E0, E1) + q0 * q1 * dot(B0, B1)) * inv;
        v[8] = (q1 * q2 * dot(E1, E2) + q1 * q2 * dot(B1, B2)) * inv;
        v[9] = (q2 * q0 * dot(E2, E0) + q2 * q0 * dot(B2, B0)) * inv;
    }
    block_store<10>(v, out);
}

// IO::SaveTransverselyIntegratedCurrents (SC/IO/SaveConfiguration.cpp:160-204): per layer
// sum_{x,y,a} of Jm^2, JmStat^2, Jp^2, JpStat^2.  K = 4.
__global__ void __launch_bounds__(256) k_currents(ObsArgs A) {
    double v[4] = {0, 0, 0, 0};
    int chunk, x, y, z;
    long s;
    double* const out = part_of<4>(A, chunk, z);
    if (!out) return;
    if (site_of(A, chunk, x, y, z, s)) {
        const int w[4] = {JM, JMS, JP, JPS};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            double j[8];
            ldv<long>(A.J, kJPlanes, 8 * w[k], s, j);
#pragma unroll
            for (int a = 0; a < 8; a++) v[k] += j[a] * j[a];
        }
    }
    block_store<4>(v, out);
}

// EnergyMomentumTensor::CreateMapBfCollision (SC/OBSERVABLES/EnergyMomentumTensor.cpp:10-77): for each
// transverse site the energy density summed over z, split at z <= (Nz - 2) / 2 (left) and above (right),
// from the elementary plaquettes of the current links and the local E.  One thread per (x, y) and chunk of
// `chunk` layers; part[(chunk * P + i) * 2 + side].  A layer's loads are a chain of their own, so the chunks are as
// short as it takes to fill the device (map_chunk): a fixed 32 layers took 183 us at 16 x 16 x 32, one block, and
// 277 us at 64 x 56 x 96.
__global__ void __launch_bounds__(256) k_tmap(ObsArgs A, double* __restrict__ part, int chunk) {
    const Geom& g = A.g;
    int pc, zc;
    if (!obs_block(A.ord, pc, zc)) return;
    const unsigned i = pc * 256u + threadIdx.x;
    if (i >= g.P) return;
    const int x = (int)(i % (unsigned)g.nx), y = (int)(i / (unsigned)g.nx);
    const int z0 = zc * chunk, z1 = min(z0 + chunk, g.nz);
    const int zsplit = (g.nz - 2) / 2;  // (zHigh - 1) / 2 with zHigh = Nz - 1
    const double ac = A.a[0] * A.a[1] * A.a[2];
    double c[3];
    for (int m = 0; m < 3; m++) c[m] = (A.a[m] / ac) * (A.a[m] / ac);  // cB = cE = (a_mu aScale^2 / aCube)^2
    const double inv_nz = 1.0 / (double)g.nz;
    double left = 0.0, right = 0.0;
    for (int z = z0; z < z1; z++) {
        const long s = i + g.P * z;
        double B[3];
        site_b2(A.U, g, x, y, z, s, B);
        const double E0 = site_e2(A.E, 0, s), E1 = site_e2(A.E, 1, s), E2 = site_e2(A.E, 2, s);
        const double t = 0.5 * (c[0] * E0 + c[1] * E1 + c[2] * E2 + c[0] * B[0] + c[1] * B[1] + c[2] * B[2]) * inv_nz;
        if (z <= zsplit) left += t; else right += t;
    }
    double* o = part + ((long)zc * g.P + i) * 2;
    o[0] = left;
    o[1] = right;
}

// layers per thread of k_tmap: up to 32, fewer until the launch has two blocks per CU
static int map_chunk(const Geom& g) {
    const long bpp = (g.P + 255) / 256;
    int chunk = 32;
    while (chunk > 1 && bpp * ((g.nz + chunk - 1) / chunk) < 512) chunk /= 2;
    return chunk;
}

// fixed-order sum of the chunks: out[i * 2 + side] = sum_c part[(c * P + i) * 2 + side]
__global__ void k_tmap_finalize(const double* __restrict__ part, double* __restrict__ out, long P, int nchunk) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 2 * P) return;
    double acc = 0.0;
#pragma unroll 8
    for (int c = 0; c < nchunk; c++) acc += part[(long)c * 2 * P + i];
    out[i] = acc;
}

// per-z finalisation: out[z*K + k] = sum_b red[(z*bpp + b)*K + k] (or max for the entries flagged in maxmask).  One
// wavefront per output: lane l adds the blocks l, l + 64, ... in order, then the lanes are added in a fixed tree, so
// the result does not depend on scheduling.  One thread per output was a chain of bpp dependent adds on strided
// loads: 107 us at 256 x 256 x 512 (bpp = 256).
//
// A block takes 16 outputs and writes them together: `out` may be host memory, where a lone 8-byte store is a transfer
// of its own.
constexpr int kFinOuts = 16;
__global__ void __launch_bounds__(64 * kFinOuts) k_finalize(const double* __restrict__ red, double* __restrict__ out,
                                                            int nz, int bpp, int K, unsigned maxmask) {
    __shared__ double sh[kFinOuts];
    const int w = threadIdx.x >> 6, i = blockIdx.x * kFinOuts + w, lane = threadIdx.x & 63;
    if (i < nz * K) {
        const int z = i / K, k = i % K;
        const bool mx = (maxmask >> k) & 1u;
        double acc = 0.0;
        for (int b = lane; b < bpp; b += 64) {
            const double v = red[((long)z * bpp + b) * K + k];
            acc = mx ? fmax(acc, v) : acc + v;
        }
        acc = mx ? wave_max(acc) : wave_sum(acc);
        if (lane == 0) sh[w] = acc;
    }
    __syncthreads();
    const int o = blockIdx.x * kFinOuts + threadIdx.x;
    if (threadIdx.x < kFinOuts && o < nz * K) out[o] = sh[threadIdx.x];
}

// ------------------------------------------------------------------------------------------------
// bitwise state checksum: sum over the physical sites' words of mix(bits ^ index-dependent key), wrapping
// 64-bit addition.  Integer addition is associative and commutative, so the result does not depend on the
// order of the per-block atomics; a change of any bit of any word changes the sum unless two 64-bit mixes
// collide.  The word index is the (plane, site) position, so permutations are detected too.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long mix64(unsigned long long z) {  // SplitMix64 finaliser (Steele et al.)
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__global__ void __launch_bounds__(256) k_checksum(const double* __restrict__ f, int NP, long S,
                                                  unsigned long long* __restrict__ out) {
    const long n = (long)NP * pad_sites(S);
    unsigned long long acc = 0;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
        // inverse of lidx: tile, plane pair, site in tile, member of the pair
        const long tile = i / ((long)NP * kTile);
        const int r = (int)(i - tile * NP * kTile);
        const long s = tile * kTile + ((r & 127) >> 1);
        if (s >= S) continue;
        const int p = 2 * (r >> 7) + (r & 1);
        const unsigned long long key = (unsigned long long)(s * NP + p) * 0x9e3779b97f4a7c15ull;
        acc += mix64((unsigned long long)__double_as_longlong(f[i]) ^ key);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) acc += __shfl_xor(acc, o, 64);
    __shared__ unsigned long long sh[4];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(out, sh[0] + sh[1] + sh[2] + sh[3]);
}

__global__ void k_zero_u64(unsigned long long* p, int n) {
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0ull;
}

// ------------------------------------------------------------------------------------------------
// Fixed device scratch of glasma_bulk_noalloc: the block partials, the per-layer sums and the 9 totals.
// Every device the library runs on holds its own copy of the array, at its own address, until the process
// ends.  Host code never passes the array's name to a kernel (on the host it only stands for the symbol):
// it uses the device address that hipGetSymbolAddress returns, looked up once per device with that device
// current.
// ------------------------------------------------------------------------------------------------
constexpr long kScratchDoubles = 1L << 20;  // 8 MiB
static __device__ __align__(256) double scratch[kScratchDoubles];
constexpr int kMaxDevices = 64;
static double* g_scratch[kMaxDevices];
static std::mutex g_scratch_mu;

static int scratch_ptr(glasma_ctx* ctx, double** out) {
    if (ctx->device < 0 || ctx->device >= kMaxDevices)
        return set_error(ctx, GLASMA_ERR_ARG, "glasma_bulk_noalloc: device ordinal out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[ctx->device]) {
        int cur = 0;
        GL_HIP(ctx, hipGetDevice(&cur));
        if (cur != ctx->device) GL_HIP(ctx, hipSetDevice(ctx->device));
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != ctx->device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return hip_fail(ctx, e, "hipGetSymbolAddress(scratch)");
        g_scratch[ctx->device] = static_cast<double*>(p);
    }
    *out = g_scratch[ctx->device];
    return 0;
}

// out[k] = the per-layer sums fin[z*K + k] added in increasing z, the order of glasma_bulk's host loop
__global__ void k_sum_layers(const double* __restrict__ fin, double* __restrict__ out, int nz, int K) {
    const int k = threadIdx.x;
    if (k >= K) return;
    double acc = 0.0;
    for (int z = 0; z < nz; z++) acc += fin[(long)z * K + k];
    out[k] = acc;
}

static int run_obs(glasma_ctx* ctx, void (*kern)(ObsArgs), int K, unsigned maxmask, std::vector<double>& per_z,
                   bool use_old) {
    const Geom& g = ctx->g;
    const int bpp = (int)((g.P + 255) / 256);
    int rc = ensure_red(ctx, (size_t)g.nz * bpp * K + (size_t)g.nz * K);
    if (rc) return rc;
    ObsArgs A;
    A.U = ctx->U[ctx->cur];
    A.UOld = use_old ? ctx->UOld : nullptr;
    A.E = ctx->E;
    A.J = ctx->J[ctx->cur];
    A.red = ctx->red;
    A.g = g;
    A.bpp = bpp;
    A.ord = obs_order(bpp, g.nz);
    for (int m = 0; m < 3; m++) A.a[m] = ctx->p.a[m];
    hipLaunchKernelGGL(kern, dim3((unsigned)(A.ord.per * kXcds)), dim3(256), 0, ctx->stream, A);
    GL_HIP(ctx, hipGetLastError());
    // results that fit go straight to pinned host memory: a copy to pageable memory is a launch, a staging copy and their
    // gaps (six records of 64 x 56 x 96 took 528 us with the copies and 472 without)
    const int n = g.nz * K;
    HostOut out(ctx, n);
    const bool direct = out.p != nullptr;
    double* fin = direct ? out.p : ctx->red + (size_t)g.nz * bpp * K;
    hipLaunchKernelGGL(k_finalize, dim3((n + kFinOuts - 1) / kFinOuts), dim3(64 * kFinOuts), 0, ctx->stream, ctx->red, fin,
                       g.nz, bpp, K, maxmask);
    GL_HIP(ctx, hipGetLastError());  // before the result is read: the memory still holds a previous record's
    per_z.resize(n);
    if (!direct)
        GL_HIP(ctx, hipMemcpyAsync(per_z.data(), fin, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    GL_HIP(ctx, hipStreamSynchronize(ctx->stream));
    out.busy = false;
    if (direct) std::memcpy(per_z.data(), fin, n * sizeof(double));
    return 0;
}

}  // namespace glasma

using namespace glasma;

// ==================================================================================================
// C ABI
// ==================================================================================================
extern "C" {

const char* glasma_version(void) { return "glasma-mi355x 0.1 (gfx950, FP64)"; }

// the message of the last failed glasma_create on this thread (there is no context to hold it)
static thread_local std::string g_create_err;

static int create_fail(int code, const std::string& msg) {
    g_create_err = msg;
    return code;
}

const char* glasma_last_error(const glasma_ctx* ctx) {
    if (!ctx) return g_create_err.c_str();
    return ctx->err.c_str();
}

int glasma_create(const glasma_params* p, glasma_ctx** out) {
    if (!p || !out) return create_fail(GLASMA_ERR_ARG, "glasma_create: null argument");
    *out = nullptr;
    if (p->nc != 3) return create_fail(GLASMA_ERR_ARG, "glasma_create: only SU(3) (nc = 3) is supported");
    for (int m = 0; m < 3; m++)
        if (p->n[m] <= 0 || !(p->a[m] > 0.0))
            return create_fail(GLASMA_ERR_ARG, "glasma_create: lattice sizes and spacings must be positive");
    if (p->bc_z != 0 && p->bc_z != 1) return create_fail(GLASMA_ERR_ARG, "glasma_create: bc_z must be 0 or 1");
    glasma_ctx* ctx = new glasma_ctx();
    stage_context_created();
    ctx->p = *p;
    ctx->g.nx = p->n[0];
    ctx->g.ny = p->n[1];
    ctx->g.nz = p->n[2];
    ctx->g.bc = p->bc_z;
    ctx->g.P = (long)p->n[0] * p->n[1];
    ctx->g.S = ctx->g.P * p->n[2];
    const long S = pad_sites(ctx->g.S);
    hipError_t e = hipGetDevice(&ctx->device);
    if (e == hipSuccess) e = hipStreamCreate(&ctx->stream);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev0);
    if (e == hipSuccess) e = hipEventCreate(&ctx->ev1);
    if (e == hipSuccess) e = hipMalloc(&ctx->U[0], (size_t)kUPlanes * S * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&ctx->U[1], (size_t)kUPlanes * S * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&ctx->UOld, (size_t)kUPlanes * S * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&ctx->E, (size_t)kEPlanes * S * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&ctx->J[0], (size_t)kJPlanes * S * sizeof(double));
    if (e == hipSuccess) e = hipMalloc(&ctx->J[1], (size_t)kJPlanes * S * sizeof(double));
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ctx->host_ev, hipEventDisableTiming);
    if (e != hipSuccess) {
        const int code = hip_code(e);
        glasma_destroy(ctx);
        return create_fail(code, std::string("glasma_create: ") + hipGetErrorString(e));
    }
    int rc = reset_fields(ctx);
    if (rc) {
        const std::string msg = std::string("glasma_create: ") + ctx->err;
        glasma_destroy(ctx);
        return create_fail(rc, msg);
    }
    g_create_err.clear();
    *out = ctx;
    return 0;
}

int glasma_destroy(glasma_ctx* ctx) {
    if (!ctx) return 0;
    if (ctx->stream) hipStreamSynchronize(ctx->stream);
    if (ctx->stream2) hipStreamSynchronize(ctx->stream2);
    double* bufs[] = {ctx->U[0], ctx->U[1], ctx->UOld, ctx->E, ctx->J[0], ctx->J[1], ctx->red, ctx->G, ctx->Gtop,
                      ctx->UG, ctx->EG, ctx->fftbuf};
    for (double* b : bufs)
        if (b) (void)hipFree(b);
    for (auto& w : ctx->wpool)
        if (w.second) (void)hipFree(w.second);
    if (ctx->ev0) hipEventDestroy(ctx->ev0);
    if (ctx->ev1) hipEventDestroy(ctx->ev1);
    if (ctx->host_ev) hipEventDestroy(ctx->host_ev);
    for (hipEvent_t ev : ctx->seg_ev)
        if (ev) hipEventDestroy(ev);
    if (ctx->stream) hipStreamDestroy(ctx->stream);
    if (ctx->stream2) hipStreamDestroy(ctx->stream2);
    delete ctx;
    stage_context_destroyed();
    return 0;
}

int glasma_release_idle(void) {
    stage_release_idle();
    return 0;
}

int glasma_memory_bytes(const glasma_ctx* ctx, size_t* bytes) {
    if (!ctx || !bytes) return GLASMA_ERR_ARG;
    const size_t S = ctx->g.S;
    size_t b = (3 * kUPlanes + kEPlanes + 2 * kJPlanes) * S * sizeof(double);
    b += ctx->red_cap * sizeof(double) + ctx->fftbuf_cap * sizeof(double);
    if (ctx->G) b += (18 * S + 18 * ctx->g.P) * sizeof(double);
    if (ctx->UG) b += kUPlanes * S * sizeof(double);
    if (ctx->EG) b += kEPlanes * S * sizeof(double);
    for (const auto& w : ctx->wpool) b += w.first * sizeof(double);
    *bytes = b;
    return 0;
}

int glasma_set_fields(glasma_ctx* ctx, const double* U, const double* E, const double* Jp, const double* Jm,
                      const double* JpStat, const double* JmStat) {
    if (!ctx) return GLASMA_ERR_ARG;
    int rc;
    if (U && (rc = upload_aos(ctx, U, ctx->U[ctx->cur], kUPlanes))) return rc;
    if (E && (rc = upload_aos(ctx, E, ctx->E, kEPlanes))) return rc;
    const double* Js[4] = {Jp, Jm, JpStat, JmStat};
    for (int w = 0; w < 4; w++)
        if (Js[w] && (rc = upload_j(ctx, Js[w], ctx->J[ctx->cur], w))) return rc;
    return 0;
}

int glasma_get_fields(glasma_ctx* ctx, double* U, double* E, double* Jp, double* Jm, double* JpStat, double* JmStat) {
    if (!ctx) return GLASMA_ERR_ARG;
    int rc;
    if (U && (rc = download_aos(ctx, ctx->U[ctx->cur], U, kUPlanes))) return rc;
    if (E && (rc = download_aos(ctx, ctx->E, E, kEPlanes))) return rc;
    double* Js[4] = {Jp, Jm, JpStat, JmStat};
    for (int w = 0; w < 4; w++)
        if (Js[w] && (rc = download_j(ctx, ctx->J[ctx->cur], Js[w], w))) return rc;
    return 0;
}

int glasma_set_uold(glasma_ctx* ctx, const double* UOld) {
    if (!ctx || !UOld) return GLASMA_ERR_ARG;
    return upload_aos(ctx, UOld, ctx->UOld, kUPlanes);
}
int glasma_get_uold(glasma_ctx* ctx, double* UOld) {
    if (!ctx || !UOld) return GLASMA_ERR_ARG;
    return download_aos(ctx, ctx->UOld, UOld, kUPlanes);
}

int glasma_get_time(const glasma_ctx* ctx, double* t, long* tsteps) {
    if (!ctx) return GLASMA_ERR_ARG;
    if (t) *t = ctx->t;
    if (tsteps) *tsteps = ctx->tsteps;
    return 0;
}
int glasma_set_time(glasma_ctx* ctx, double t, long tsteps) {
    if (!ctx) return GLASMA_ERR_ARG;
    ctx->t = t;
    ctx->tsteps = tsteps;
    return 0;
}

int glasma_update_async(glasma_ctx* ctx, int nsteps) {
    if (!ctx || nsteps < 0) return GLASMA_ERR_ARG;
    if (nsteps == 0) return 0;
    GL_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
    for (int i = 0; i < nsteps; i++) {
        launch_step(ctx, i == nsteps - 1);
        ctx->tsteps++;
        ctx->t += ctx->p.dt;
    }
    GL_HIP(ctx, hipGetLastError());
    GL_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    ctx->last_step_ms = -(double)nsteps;  // resolved by glasma_last_step_kernel_ms
    return 0;
}

int glasma_synchronize(glasma_ctx* ctx) {
    if (!ctx) return GLASMA_ERR_ARG;
    GL_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

int glasma_update(glasma_ctx* ctx, int nsteps) {
    int rc = glasma_update_async(ctx, nsteps);
    if (rc) return rc;
    return glasma_synchronize(ctx);
}

int glasma_last_step_kernel_ms(const glasma_ctx* ctx, double* ms) {
    if (!ctx || !ms) return GLASMA_ERR_ARG;
    glasma_ctx* c = const_cast<glasma_ctx*>(ctx);
    if (c->last_step_ms < 0) {
        const double n = -c->last_step_ms;
        float el = 0.f;
        GL_HIP(c, hipEventSynchronize(c->ev1));
        GL_HIP(c, hipEventElapsedTime(&el, c->ev0, c->ev1));
        c->last_step_ms = (double)el / n;
    }
    *ms = c->last_step_ms;
    return 0;
}

int glasma_fill_random(glasma_ctx* ctx, unsigned long seed, double link_scale, double e_scale, double j_scale) {
    if (!ctx) return GLASMA_ERR_ARG;
    const long S = ctx->g.S;
    hipLaunchKernelGGL(k_fill_random, dim3((unsigned)((S + 255) / 256)), dim3(256), 0, ctx->stream, ctx->U[ctx->cur],
                       ctx->E, ctx->J[ctx->cur], S, (unsigned long long)seed, link_scale, e_scale, j_scale);
    GL_HIP(ctx, hipGetLastError());
    GL_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

int glasma_bulk(glasma_ctx* ctx, double* out9) {
    if (!ctx || !out9) return GLASMA_ERR_ARG;
    std::vector<double> pz;
    int rc = run_obs(ctx, k_bulk, 9, 0u, pz, false);
    if (rc) return rc;
    for (int k = 0; k < 9; k++) out9[k] = 0.0;
    for (int z = 0; z < ctx->g.nz; z++)
        for (int k = 0; k < 9; k++) out9[k] += pz[(size_t)z * 9 + k];
    for (int k = 0; k < 9; k++)
        if (!std::isfinite(out9[k]))
            return set_error(ctx, GLASMA_ERR_NUMERIC, "non-finite fields: the evolution diverged or a step's current "
                                                      "hand-over timed out (sums returned as computed)");
    return 0;
}

int glasma_bulk_noalloc(glasma_ctx* ctx, double* out9) {
    if (!ctx || !out9) return GLASMA_ERR_ARG;
    const Geom& g = ctx->g;
    const int bpp = (int)((g.P + 255) / 256);
    const long need = (long)g.nz * bpp * 9 + (long)g.nz * 9 + 9;
    if (need > kScratchDoubles) {
        char msg[200];
        std::snprintf(msg, sizeof(msg), "glasma_bulk_noalloc: this lattice needs %ld doubles of scratch, more than the "
                      "fixed %ld (use glasma_bulk)", need, kScratchDoubles);
        return set_error(ctx, GLASMA_ERR_ARG, msg);
    }
    double* ptr = nullptr;
    int rc = scratch_ptr(ctx, &ptr);
    if (rc) return rc;
    // the kernels write every entry they later read (all blocks store their partials), so nothing is cleared
    ObsArgs A;
    A.U = ctx->U[ctx->cur];
    A.UOld = nullptr;
    A.E = ctx->E;
    A.J = ctx->J[ctx->cur];
    A.red = ptr;
    A.g = g;
    A.bpp = bpp;
    A.ord = obs_order(bpp, g.nz);
    for (int m = 0; m < 3; m++) A.a[m] = ctx->p.a[m];
    double* fin = ptr + (long)g.nz * bpp * 9;
    double* tot = fin + (long)g.nz * 9;
    hipLaunchKernelGGL(k_bulk, dim3((unsigned)(A.ord.per * kXcds)), dim3(256), 0, ctx->stream, A);
    hipLaunchKernelGGL(k_finalize, dim3((g.nz * 9 + kFinOuts - 1) / kFinOuts), dim3(64 * kFinOuts), 0, ctx->stream, ptr, fin,
                       g.nz, bpp, 9, 0u);
    hipLaunchKernelGGL(k_sum_layers, dim3(1), dim3(64), 0, ctx->stream, fin, tot, g.nz, 9);
    GL_HIP(ctx, hipGetLastError());
    GL_HIP(ctx, hipMemcpyAsync(out9, tot, 9 * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    GL_HIP(ctx, hipStreamSynchronize(ctx->stream));
    for (int k = 0; k < 9; k++)
        if (!std::isfinite(out9[k]))
            return set_error(ctx, GLASMA_ERR_NUMERIC, "non-finite fields: the evolution diverged or a step's current "
                                                      "hand-over timed out (sums returned as computed)");
    return 0;
}

int glasma_gauss(glasma_ctx* ctx, double* per_z, double* gmax, double* grms) {
    if (!ctx) return GLASMA_ERR_ARG;
    std::vector<double> pz;
    int rc = run_obs(ctx, k_gauss, 2, 2u, pz, false);
    if (rc) return rc;
    double sq = 0.0, mx = 0.0;
    for (int z = 0; z < ctx->g.nz; z++) {
        if (per_z) per_z[z] = pz[2 * z] / (double)ctx->g.P;
        sq += pz[2 * z];
        mx = fmax(mx, pz[2 * z + 1]);
    }
    if (gmax) *gmax = mx;
    if (grms) *grms = sqrt(sq / (8.0 * (double)ctx->g.S));
    return 0;
}

int glasma_unitarity(glasma_ctx* ctx, double* umax, double* urms) {
    if (!ctx) return GLASMA_ERR_ARG;
    std::vector<double> pz;
    int rc = run_obs(ctx, k_unitarity, 2, 2u, pz, false);
    if (rc) return rc;
    double sq = 0.0, mx = 0.0;
    for (int z = 0; z < ctx->g.nz; z++) {
        sq += pz[2 * z];
        mx = fmax(mx, pz[2 * z + 1]);
    }
    if (umax) *umax = mx;
    if (urms) *urms = sqrt(sq / (3.0 * (double)ctx->g.S));
    return 0;
}

int glasma_checksum(glasma_ctx* ctx, uint64_t* out4) {
    if (!ctx || !out4) return GLASMA_ERR_ARG;
    int rc = ensure_red(ctx, 4);
    if (rc) return rc;
    unsigned long long* acc = reinterpret_cast<unsigned long long*>(ctx->red);
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, ctx->stream, acc, 4);
    const double* fields[4] = {ctx->U[ctx->cur], ctx->UOld, ctx->E, ctx->J[ctx->cur]};
    const int np[4] = {kUPlanes, kUPlanes, kEPlanes, kJPlanes};
    for (int k = 0; k < 4; k++) {
        const long n = (long)np[k] * pad_sites(ctx->g.S);
        const unsigned nb = (unsigned)std::min<long>(4096, (n + 255) / 256);
        hipLaunchKernelGGL(k_checksum, dim3(nb), dim3(256), 0, ctx->stream, fields[k], np[k], ctx->g.S, acc + k);
    }
    GL_HIP(ctx, hipGetLastError());
    unsigned long long h[4];
    GL_HIP(ctx, hipMemcpyAsync(h, acc, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
    GL_HIP(ctx, hipStreamSynchronize(ctx->stream));
    for (int k = 0; k < 4; k++) out4[k] = h[k];
    return 0;
}

int glasma_emt(glasma_ctx* ctx, double* out) {
    if (!ctx || !out) return GLASMA_ERR_ARG;
    std::vector<double> pz;
    int rc = run_obs(ctx, k_emt, 10, 0u, pz, true);
    if (rc) return rc;
    std::memcpy(out, pz.data(), pz.size() * sizeof(double));
    return 0;
}

int glasma_field_profile(glasma_ctx* ctx, double* out) {
    if (!ctx || !out) return GLASMA_ERR_ARG;
    std::vector<double> pz;
    int rc = run_obs(ctx, k_bulk, 9, 0u, pz, false);
    if (rc) return rc;
    const double inv = 1.0 / (double)ctx->g.P;
    for (int z = 0; z < ctx->g.nz; z++) {
        const double* r = &pz[(size_t)z * 9];  // E0^2 E1^2 E2^2 B0 B1 B2 (sums over the layer)
        out[4 * z + 0] = 0.5 * (r[3] * inv + r[4] * inv);
        out[4 * z + 1] = 0.5 * (r[5] * inv);
        out[4 * z + 2] = 0.5 * (r[0] * inv + r[1] * inv);
        out[4 * z + 3] = 0.5 * (r[2] * inv);
    }
    return 0;
}

int glasma_current_profile(glasma_ctx* ctx, double* out) {
    if (!ctx || !out) return GLASMA_ERR_ARG;
    std::vector<double> pz;
    int rc = run_obs(ctx, k_currents, 4, 0u, pz, false);
    if (rc) return rc;
    const int nz = ctx->g.nz;
    const double inv = 1.0 / (double)ctx->g.P;
    // rows z = -1 .. nz; the ghost layers hold what SynchronizeGhostCells puts there
    for (int r = 0; r < nz + 2; r++) {
        const int z = r - 1;
        const int src = z < 0 ? (ctx->g.bc ? nz - 1 : 0) : (z >= nz ? (ctx->g.bc ? 0 : nz - 1) : z);
        for (int k = 0; k < 4; k++) out[4 * r + k] = 0.5 * pz[(size_t)src * 4 + k] * inv;
    }
    return 0;
}

int glasma_transverse_energy_map(glasma_ctx* ctx, double* out) {
    if (!ctx || !out) return GLASMA_ERR_ARG;
    const Geom& g = ctx->g;
    const int bpp = (int)((g.P + 255) / 256);
    const int chunk = map_chunk(g), nchunk = (g.nz + chunk - 1) / chunk;
    int rc = ensure_red(ctx, (size_t)(nchunk + 1) * 2 * g.P);
    if (rc) return rc;
    ObsArgs A;
    A.U = ctx->U[ctx->cur];
    A.UOld = nullptr;
    A.E = ctx->E;
    A.J = ctx->J[ctx->cur];
    A.red = nullptr;
    A.g = g;
    A.bpp = bpp;
    A.ord = obs_order(bpp, nchunk);
    for (int m = 0; m < 3; m++) A.a[m] = ctx->p.a[m];
    HostOut host(ctx, 2 * g.P);
    const bool direct = host.p != nullptr;
    double* fin = direct ? host.p : ctx->red + (size_t)nchunk * 2 * g.P;
    hipLaunchKernelGGL(k_tmap, dim3((unsigned)(A.ord.per * kXcds)), dim3(256), 0, ctx->stream, A, ctx->red, chunk);
    hipLaunchKernelGGL(k_tmap_finalize, dim3((unsigned)((2 * g.P + 255) / 256)), dim3(256), 0, ctx->stream, ctx->red,
                       fin, (long)g.P, nchunk);
    GL_HIP(ctx, hipGetLastError());
    if (!direct) GL_HIP(ctx, hipMemcpyAsync(out, fin, 2 * g.P * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    GL_HIP(ctx, hipStreamSynchronize(ctx->stream));
    host.busy = false;
    if (direct) std::memcpy(out, fin, 2 * g.P * sizeof(double));
    return 0;
}

}  // extern "C"
