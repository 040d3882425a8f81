// In-LDS FFT core shared by the transform passes (fft.hip) and the kernels that fuse a transform of their own x lines
// (gauge.hip): line factorisation, complex helpers and the self-sorting Stockham stages over lines held in LDS.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>

namespace glasma {

constexpr int kMaxStages = 24;
constexpr int kMaxGenericRadix = 16;

struct Radices {
    int n, nst;
    int r[kMaxStages];
};

inline int factorize(int n, Radices& R) {
    R.n = n;
    R.nst = 0;
    int m = n;
    for (int f : {4, 2, 3}) {
        while (m % f == 0) {
            if (R.nst == kMaxStages) return -1;
            R.r[R.nst++] = f;
            m /= f;
        }
    }
    for (int p = 5; m > 1; p += 2) {
        while (m % p == 0) {
            if (p > kMaxGenericRadix || R.nst == kMaxStages) return -1;
            R.r[R.nst++] = p;
            m /= p;
        }
    }
    return 0;
}

// the odd primes that a line's stages need (stockham)
inline int odd_level(const Radices& R) {
    int l = 0;
    for (int k = 0; k < R.nst; k++) l = std::max(l, R.r[k] > 7 ? 2 : R.r[k] > 3 && R.r[k] != 4 ? 1 : 0);
    return l;
}

typedef double dbl2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ dbl2 cmul(dbl2 a, dbl2 b) { return dbl2{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
// twiddle exp(sign * 2 pi i k / n) from the forward table
__device__ __forceinline__ dbl2 twid(const dbl2* tw, int k, int sign) {
    dbl2 w = tw[k];
    return sign < 0 ? w : dbl2{w.x, -w.y};
}
// the same from a two-level table of kTwSplit + ceil(n / kTwSplit) entries: lo[j] = exp(-2 pi i j / n), j < kTwSplit,
// then hi[j] = exp(-2 pi i kTwSplit j / n); exp(-2 pi i k / n) = lo[k % kTwSplit] hi[k / kTwSplit], within two units
// of the last place.  1.5 KiB for a line of 2048, where the full table takes 32 KiB of LDS.
constexpr int kTwSplit = 32;
__device__ __forceinline__ dbl2 twid_split(const dbl2* tw, int k, int sign) {
    dbl2 w = cmul(tw[k & (kTwSplit - 1)], tw[kTwSplit + k / kTwSplit]);
    return sign < 0 ? w : dbl2{w.x, -w.y};
}
template <bool SPLIT>
__device__ __forceinline__ dbl2 twiddle(const dbl2* tw, int k, int sign) {
    return SPLIT ? twid_split(tw, k, sign) : twid(tw, k, sign);
}

// a / d for 0 <= a < 2^20 and 1 <= d < 2^20, with rd = 1/d in FP32: the FP32 product is within 1/8 of a / d,
// so the truncated estimate is off by at most one, and one remainder test corrects it.  The index arithmetic
// below divides by run-time lengths once per element; this replaces the integer division sequence.
__device__ __forceinline__ int qdiv(int a, int d, float rd) {
    int q = (int)((float)a * rd);
    const int r = a - q * d;
    if (r < 0) q--;
    else if (r >= d) q++;
    return q;
}

// DFT of odd prime length R in registers, in place and in order: with s_m = v_m + v_(R-m) and d_m = v_m - v_(R-m), m <=
// (R-1)/2, V_k = v_0 + sum_m cos(2 pi k m / R) s_m + i sign sum_m sin(2 pi k m / R) d_m, and V_(R-k) with the other sign
template <int R>
struct OddRoots;
template <>
struct OddRoots<5> {
    static constexpr double c[3] = {1.0, 0.30901699437494742410, -0.80901699437494742410};
    static constexpr double s[3] = {0.0, 0.95105651629515357212, 0.58778525229247312917};
};
template <>
struct OddRoots<7> {
    static constexpr double c[4] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
    static constexpr double s[4] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
};
template <>
struct OddRoots<11> {
    static constexpr double c[6] = {1.0, 0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                                -0.65486073394528506406, -0.95949297361449738989};
    static constexpr double s[6] = {0.0, 0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
                                0.75574957435425828377, 0.28173255684142969771};
};
template <>
struct OddRoots<13> {
    static constexpr double c[7] = {1.0, 0.88545602565320989590, 0.56806474673115580251, 0.12053668025532305335,
                                -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716};
    static constexpr double s[7] = {0.0, 0.46472317204376854566, 0.82298386589365639458, 0.99270887409805399280,
                                0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715};
};
template <int R>
__device__ __forceinline__ void odd_dft(dbl2* v, int sign) {
    constexpr int H = (R - 1) / 2;
    dbl2 s[H], d[H];
    const dbl2 v0 = v[0];
#pragma unroll
    for (int m = 1; m <= H; m++) {
        s[m - 1] = v[m] + v[R - m];
        d[m - 1] = v[m] - v[R - m];
        v[0] += s[m - 1];
    }
#pragma unroll
    for (int k = 1; k <= H; k++) {
        dbl2 a = v0, b = dbl2{0.0, 0.0};
#pragma unroll
        for (int m = 1; m <= H; m++) {
            const int e = (k * m) % R, f = e <= H ? e : R - e;
            a += OddRoots<R>::c[f] * s[m - 1];
            b += (e <= H ? OddRoots<R>::s[f] : -OddRoots<R>::s[f]) * d[m - 1];
        }
        const dbl2 q = sign < 0 ? dbl2{b.y, -b.x} : dbl2{-b.y, b.x};  // sign i b
        v[k] = a + q;
        v[R - k] = a - q;
    }
}

// the forward twiddle table exp(-2 pi i j / n), j < n, of the current device (fft.hip; kept for the process lifetime)
hipError_t fft_twiddles(int n, const dbl2** out);
// the two-level table of twid_split, the same way
hipError_t fft_twiddles_split(int n, const dbl2** out);
// the factorisation of a line of length n with the refusals of every transform here (above 2048, a prime factor above
// 13: an error code, the reason in fft_last_error)
int fft_radices(int n, Radices& R);
// LDS a workgroup may ask for on the current device (160 KiB on gfx950 where the runtime grants it)
hipError_t fft_lds_limit(size_t* out);
// entries of the two-level table of twid_split
__host__ __device__ inline int split_entries(int n) { return kTwSplit + (n + kTwSplit - 1) / kTwSplit; }

// one butterfly of odd prime radix R of a Stockham stage (see stockham): the inputs once from LDS, in registers
template <int R, bool SPLIT>
__device__ __forceinline__ void odd_stage(const dbl2* al, dbl2* bl, int j, int nr, int k, int tstride, int od, int Ns,
                                          int sign, const dbl2* tw, int es) {
    dbl2 v[R];
#pragma unroll
    for (int q = 0; q < R; q++) v[q] = al[(j + q * nr) * es];
    if (k) {
#pragma unroll
        for (int q = 1; q < R; q++) v[q] = cmul(v[q], twiddle<SPLIT>(tw, k * q * tstride, sign));
    }
    odd_dft<R>(v, sign);
#pragma unroll
    for (int q = 0; q < R; q++) bl[(od + q * Ns) * es] = v[q];
}

// The Stockham stages over the lpb lines in buffer `cur` (line li at lb + cur * bs + li * ld); buffer c starts at
// lb + c * bs.  Returns which buffer holds the transform.  The buffers are addressed as offsets from the LDS base, not through
// a run-time indexed pointer array, so the compiler keeps them in the LDS address space (ds_read / ds_write);
// a generic pointer would give flat instructions, whose waits also wait for every global load in flight.
// Every stage ends with a barrier.  Elements of a line lie es apart.
// ODD: the odd primes compiled in (odd_level(R)): 0 for lengths 2^a 3^b, 1 with 5 and 7, 2 with 11 and 13 as well.  Each
// takes its inputs into registers once (a direct DFT that read LDS R^2 times took 72 us for a pass of length 100 at
// 100 x 100 x 100, this 38; the filtered pass 239 and 95; of length 91 at 88 x 78 x 91 405 and 86), and the registers
// that takes cost lengths without such factors (pass of length 128 at 128 x 128 x 256: 131 us against 125), hence levels.
template <bool SPLIT = false, int ODD = 0>
__device__ __forceinline__ int stockham(dbl2* const lb, int bs, int cur, const Radices& R, int lpb, int ld,
                                        int sign, const dbl2* tw, int es = 1) {
    const int n = R.n;
    int Ns = 1;
    for (int st = 0; st < R.nst; st++) {
        const int r = R.r[st];
        const int nr = n / r;
        const int tstride = n / (Ns * r);
        const dbl2* a = lb + cur * bs;
        dbl2* b = lb + (cur ^ 1) * bs;
        const float rnr = 1.0f / (float)nr, rns = 1.0f / (float)Ns;
        for (int it = threadIdx.x; it < lpb * nr; it += blockDim.x) {
            const int li = qdiv(it, nr, rnr);
            const int j = it - li * nr;
            const int jq = qdiv(j, Ns, rns);
            const int k = j - jq * Ns;
            const dbl2* al = a + li * ld;
            dbl2* bl = b + li * ld;
            const int od = jq * Ns * r + k;
            if (r == 4) {
                dbl2 v0 = al[j * es], v1 = al[(j + nr) * es], v2 = al[(j + 2 * nr) * es], v3 = al[(j + 3 * nr) * es];
                if (k) {
                    v1 = cmul(v1, twiddle<SPLIT>(tw, k * tstride, sign));
                    v2 = cmul(v2, twiddle<SPLIT>(tw, 2 * k * tstride, sign));
                    v3 = cmul(v3, twiddle<SPLIT>(tw, 3 * k * tstride, sign));
                }
                dbl2 t0 = v0 + v2, t1 = v0 - v2, t2 = v1 + v3, d = v1 - v3;
                // t3 = (sign * i) * d
                dbl2 t3 = sign < 0 ? dbl2{d.y, -d.x} : dbl2{-d.y, d.x};
                bl[od * es] = t0 + t2;
                bl[(od + Ns) * es] = t1 + t3;
                bl[(od + 2 * Ns) * es] = t0 - t2;
                bl[(od + 3 * Ns) * es] = t1 - t3;
            } else if (r == 2) {
                dbl2 v0 = al[j * es], v1 = al[(j + nr) * es];
                if (k) v1 = cmul(v1, twiddle<SPLIT>(tw, k * tstride, sign));
                bl[od * es] = v0 + v1;
                bl[(od + Ns) * es] = v0 - v1;
            } else if (r == 3) {
                dbl2 v0 = al[j * es], v1 = al[(j + nr) * es], v2 = al[(j + 2 * nr) * es];
                if (k) {
                    v1 = cmul(v1, twiddle<SPLIT>(tw, k * tstride, sign));
                    v2 = cmul(v2, twiddle<SPLIT>(tw, 2 * k * tstride, sign));
                }
                const double h = 0.86602540378443864676;  // sqrt(3)/2
                dbl2 t = v1 + v2, d = v1 - v2;
                dbl2 m = v0 - 0.5 * t;
                // (sign * i * h) * d
                dbl2 q = sign < 0 ? dbl2{h * d.y, -h * d.x} : dbl2{-h * d.y, h * d.x};
                bl[od * es] = v0 + t;
                bl[(od + Ns) * es] = m + q;
                bl[(od + 2 * Ns) * es] = m - q;
            } else if (ODD >= 1 && r == 5) {
                odd_stage<5, SPLIT>(al, bl, j, nr, k, tstride, od, Ns, sign, tw, es);
            } else if (ODD >= 1 && r == 7) {
                odd_stage<7, SPLIT>(al, bl, j, nr, k, tstride, od, Ns, sign, tw, es);
            } else if (ODD >= 2 && r == 11) {
                odd_stage<11, SPLIT>(al, bl, j, nr, k, tstride, od, Ns, sign, tw, es);
            } else if (ODD >= 2 && r == 13) {
                odd_stage<13, SPLIT>(al, bl, j, nr, k, tstride, od, Ns, sign, tw, es);
            }
        }
        __syncthreads();
        cur ^= 1;
        Ns *= r;
    }
    return cur;
}

}  // namespace glasma
