// Field transfer between host arrays in the reference's array-of-structs layout and the tiled device layout.
//
// The host arrays are ordinary (pageable) memory, which the device cannot reach.  A transfer is cut into pieces of up to
// 1 MiB; each of up to 8 workers takes the next piece, transposes it on the device straight from or into its own pinned
// buffer (one kernel on its own stream, the buffer read or written over the host link) and copies it from or to the host
// array, so that the link and the copies run at the same time and a fresh array's pages are touched by several threads.
// One copy through the runtime's own staging, with a device-side intermediate, moved 13 GB/s (48 x 48 x 96 fields in, ten
// steps and fields out: 29 ms).
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>

#include "internal.h"

namespace glasma {

namespace {

constexpr size_t kPiece = 1 << 20;
constexpr int kWorkers = 8;

// the pinned buffers and streams of one transfer
struct StageSet {
    int device = -1;
    double* buf[kWorkers] = {};
    hipStream_t stream[kWorkers] = {};
};

// Sets not in use: at most kIdleSets (for that many threads at once) while the process holds contexts, one after that,
// until glasma_release_idle.  A set costs 2 to 12 ms to make and give back (pinning 8 MiB, eight streams), more than small
// fields take, so contexts made one after another and threads side by side have to find theirs again.  A context with its
// fields set and read took 2.8 ms at 16 x 16 x 32 and 13.6 to 16 at 32 x 32 x 64 when the last context took the sets with
// it (1.8 and 13.4 through the runtime's own staging), 1.05 and 7.5 now; eight threads with two idle sets between them 0.69
// ms for set and get at 16 x 16 x 32, 0.35 now.
constexpr int kIdleSets = 8;
std::mutex g_mu;
StageSet* g_idle[kIdleSets] = {};
int g_contexts = 0;

// the same for the memory of small results (HostOut, 64 KiB each)
struct ResultBlock {
    int device = -1;
    double* p = nullptr;
};
ResultBlock g_results[kIdleSets];

void destroy_set(StageSet* s) {
    for (int w = 0; w < kWorkers; w++) {
        if (s->stream[w]) (void)hipStreamDestroy(s->stream[w]);
        if (s->buf[w]) (void)hipHostFree(s->buf[w]);
    }
    delete s;
}

// a set for the current device with the buffers of up to *workers workers (fewer where no more memory can be pinned)
hipError_t acquire_set(int device, int* workers, StageSet** out) {
    StageSet* s = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (StageSet*& i : g_idle)
            if (!s && i && i->device == device) std::swap(s, i);
    }
    if (!s) {
        s = new (std::nothrow) StageSet();
        if (!s) return hipErrorOutOfMemory;
        s->device = device;
    }
    hipError_t e = hipSuccess;
    int n = 0;
    for (; n < *workers; n++) {
        if (!s->buf[n]) e = hipHostMalloc(reinterpret_cast<void**>(&s->buf[n]), kPiece, hipHostMallocDefault);
        if (e == hipSuccess && !s->stream[n]) e = hipStreamCreate(&s->stream[n]);
        if (e != hipSuccess) break;
    }
    if (n == 0) {
        destroy_set(s);
        return e;
    }
    if (e != hipSuccess) (void)hipGetLastError();
    *workers = n;
    *out = s;
    return hipSuccess;
}

void release_set(StageSet* s) {
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (StageSet*& i : g_idle)
            if (s && !i && g_contexts > 0) std::swap(s, i);
    }
    if (s) destroy_set(s);
}

// One tile (64 sites) per block: R doubles per site (planes p0 .. p0+R-1 of a field with NP planes) between the tiled
// device field and n sites of an array of records, through LDS so that both sides move 16 bytes per lane in order.
constexpr int kMaxRecord = kUPlanes;
constexpr int kRecordPad = 2;  // 16-byte columns of a record fall on different banks for neighbouring sites

template <bool TO_DEVICE>
__global__ void __launch_bounds__(256) k_transpose(double* __restrict__ soa, double* __restrict__ aos, long first, long n, int R,
                                                   int NP, int p0) {
    __shared__ __align__(16) double sh[kTile * (kMaxRecord + kRecordPad)];
    const int W = R / 2, ld = R + kRecordPad;
    const long t0 = (long)blockIdx.x * kTile;
    const int m = (int)(n - t0 < kTile ? n - t0 : kTile);
    d2_t* f = reinterpret_cast<d2_t*>(soa) + ((first + t0) / kTile * (NP >> 1) + (p0 >> 1)) * kTile;
    d2_t* r = reinterpret_cast<d2_t*>(aos) + t0 * W;
    if (TO_DEVICE) {
        for (int i = threadIdx.x; i < m * W; i += 256) *reinterpret_cast<d2_t*>(sh + i / W * ld + 2 * (i % W)) = r[i];
        __syncthreads();
        for (int i = threadIdx.x; i < W * kTile; i += 256)
            if (i % kTile < m) f[i] = *reinterpret_cast<d2_t*>(sh + i % kTile * ld + 2 * (i / kTile));
    } else {
        for (int i = threadIdx.x; i < W * kTile; i += 256)
            if (i % kTile < m) *reinterpret_cast<d2_t*>(sh + i % kTile * ld + 2 * (i / kTile)) = f[i];
        __syncthreads();
        for (int i = threadIdx.x; i < m * W; i += 256) r[i] = *reinterpret_cast<d2_t*>(sh + i / W * ld + 2 * (i % W));
    }
}

// host: the S records of the lattice (no ghosts)
template <bool TO_DEVICE>
int transfer(glasma_ctx* ctx, double* host, double* soa, int R, int NP, int p0) {
    const long S = ctx->g.S;
    const long per = (long)(kPiece / (R * sizeof(double))) / kTile * kTile;  // whole tiles
    const long npiece = (S + per - 1) / per;
    GL_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const unsigned hc = std::thread::hardware_concurrency();
    int workers = (int)std::min<long>(npiece, std::min<long>(kWorkers, hc > 2 ? hc : 2));
    int current = ctx->device;
    GL_HIP(ctx, hipGetDevice(&current));
    if (current != ctx->device) GL_HIP(ctx, hipSetDevice(ctx->device));
    StageSet* set = nullptr;
    hipError_t e0 = acquire_set(ctx->device, &workers, &set);
    if (e0 != hipSuccess) {
        if (current != ctx->device) (void)hipSetDevice(current);
        return hip_fail(ctx, e0, "pinned buffers of a field transfer");
    }
    std::atomic<long> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](int w) {
        hipError_t e = w ? hipSetDevice(ctx->device) : hipSuccess;
        for (long k; e == hipSuccess && failed.load() == (int)hipSuccess && (k = next.fetch_add(1)) < npiece;) {
            const long s0 = k * per, n = std::min(per, S - s0);
            double* h = host + (size_t)s0 * R;
            const size_t bytes = (size_t)n * R * sizeof(double);
            if (TO_DEVICE) std::memcpy(set->buf[w], h, bytes);
            hipLaunchKernelGGL(k_transpose<TO_DEVICE>, dim3((unsigned)((n + kTile - 1) / kTile)), dim3(256), 0, set->stream[w],
                               soa, set->buf[w], s0, n, R, NP, p0);
            e = hipGetLastError();
            if (e == hipSuccess) e = hipStreamSynchronize(set->stream[w]);
            if (!TO_DEVICE && e == hipSuccess) std::memcpy(h, set->buf[w], bytes);
        }
        if (e != hipSuccess) failed.store((int)e);
    };
    std::thread th[kWorkers];
    for (int w = 1; w < workers; w++) {
        try {
            th[w] = std::thread(work, w);
        } catch (const std::exception&) {
            break;  // the workers that run take its pieces
        }
    }
    work(0);
    for (std::thread& t : th)
        if (t.joinable()) t.join();
    const hipError_t e = (hipError_t)failed.load();
    if (e != hipSuccess)  // a kernel may still be using a buffer
        for (int w = 0; w < workers; w++) (void)hipStreamSynchronize(set->stream[w]);
    release_set(set);
    if (current != ctx->device) (void)hipSetDevice(current);
    if (e != hipSuccess) return hip_fail(ctx, e, TO_DEVICE ? "upload_aos" : "download_aos");
    return 0;
}

}  // namespace

void stage_context_created() {
    std::lock_guard<std::mutex> lock(g_mu);
    g_contexts++;
}
// gives the sets and result blocks not in use back, all but `keep` of each
static void release_idle(int keep) {
    StageSet* sets[kIdleSets] = {};
    ResultBlock results[kIdleSets];
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (int i = 0, n = 0; i < kIdleSets; i++)
            if (g_idle[i] && n++ >= keep) std::swap(sets[i], g_idle[i]);
        for (int i = 0, n = 0; i < kIdleSets; i++)
            if (g_results[i].p && n++ >= keep) std::swap(results[i], g_results[i]);
    }
    for (StageSet* s : sets)
        if (s) destroy_set(s);
    for (const ResultBlock& r : results)
        if (r.p) (void)hipHostFree(r.p);
}
void stage_context_destroyed() {
    bool last;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        last = --g_contexts == 0;
    }
    if (last) release_idle(1);
}
void stage_release_idle() { release_idle(0); }

HostOut::HostOut(const glasma_ctx* ctx, long doubles) : ctx_(ctx) {
    if (doubles > kHostOut) return;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (ResultBlock& r : g_results)
            if (!p && r.p && r.device == ctx->device) std::swap(p, r.p);
    }
    if (!p && hipHostMalloc(reinterpret_cast<void**>(&p), kHostOut * sizeof(double), hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        p = nullptr;
    }
}
HostOut::~HostOut() {
    if (!p) return;
    if (busy) (void)hipStreamSynchronize(ctx_->stream);
    {
        std::lock_guard<std::mutex> lock(g_mu);
        for (ResultBlock& r : g_results)
            if (p && !r.p) {
                std::swap(p, r.p);
                r.device = ctx_->device;
            }
    }
    if (p) (void)hipHostFree(p);
}

int upload_aos(glasma_ctx* ctx, const double* host_with_ghosts, double* dev_soa, int R, int NP, int p0) {
    return transfer<true>(ctx, const_cast<double*>(host_with_ghosts) + (size_t)ctx->g.P * R, dev_soa, R, NP < 0 ? R : NP, p0);
}

// fill the two ghost layers of a host AoS array as SynchronizeGhostCells does
void host_sync_ghosts(const glasma_ctx* ctx, double* h, int R) {
    const long P = ctx->g.P * R;
    const int nz = ctx->g.nz;
    if (ctx->p.bc_z == 0) {
        std::memcpy(h, h + P, P * sizeof(double));
        std::memcpy(h + (long)(nz + 1) * P, h + (long)nz * P, P * sizeof(double));
    } else {
        std::memcpy(h, h + (long)nz * P, P * sizeof(double));
        std::memcpy(h + (long)(nz + 1) * P, h + P, P * sizeof(double));
    }
}

int download_aos(glasma_ctx* ctx, const double* dev_soa, double* host_with_ghosts, int R, int NP, int p0) {
    const int rc = transfer<false>(ctx, host_with_ghosts + (size_t)ctx->g.P * R, const_cast<double*>(dev_soa), R,
                                   NP < 0 ? R : NP, p0);
    if (rc) return rc;
    host_sync_ghosts(ctx, host_with_ghosts, R);
    return 0;
}

}  // namespace glasma
