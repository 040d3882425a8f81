// A stand-in for the HIP runtime, for tests of the library's host code on machines without a GPU: device memory is host
// memory, copies are copies, kernels do nothing.  A test can refuse the n-th kernel launch and allocations beyond a
// limit, and read how often the runtime was asked for memory, streams and launches, and of which kernels.  Loaded with
// RTLD_GLOBAL before libglasma.so, its functions take the place of the runtime's there.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {
std::mutex mu;
std::map<void*, size_t> device, pinned;
std::map<const void*, std::string> kernels;  // device names of the registered kernels
std::map<std::string, long> launched;
long launches, refuse = -1, streams, pins, transfers_h2d, transfers_d2h;
size_t limit = (size_t)288 << 30, shown, used, pin_limit = ~(size_t)0, pinned_bytes;
thread_local hipError_t last = hipSuccess;
hipError_t fail(hipError_t e) { return last = e; }
hipError_t get(std::map<void*, size_t>& m, size_t& total, size_t cap, void** p, size_t n) {
    std::lock_guard<std::mutex> lock(mu);
    if (n > cap || total > cap - n) return fail(hipErrorOutOfMemory);
    *p = std::calloc(1, n ? n : 1);
    if (!*p) return fail(hipErrorOutOfMemory);
    m[*p] = n;
    total += n;
    return hipSuccess;
}
hipError_t put(std::map<void*, size_t>& m, size_t& total, void* p) {
    std::lock_guard<std::mutex> lock(mu);
    if (!p) return hipSuccess;
    auto it = m.find(p);
    if (it == m.end()) return fail(hipErrorInvalidValue);
    total -= it->second;
    m.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t copy(void* d, const void* s, size_t n, hipMemcpyKind k) {
    std::memcpy(d, s, n);
    std::lock_guard<std::mutex> lock(mu);
    transfers_h2d += k == hipMemcpyHostToDevice;
    transfers_d2h += k == hipMemcpyDeviceToHost;
    return hipSuccess;
}
template <class T>
T handle() {
    static long next = 0;
    std::lock_guard<std::mutex> lock(mu);
    return reinterpret_cast<T>((next += 16) + 4096);
}
thread_local dim3 cfg_grid, cfg_block;
thread_local size_t cfg_lds;
thread_local hipStream_t cfg_stream;
}  // namespace

extern "C" {
// controls
void fake_refuse_launch(long n) { refuse = n < 0 ? -1 : launches + n; }  // the n-th launch from now on
void fake_limit(size_t bytes) { limit = bytes; }
void fake_show(size_t bytes) { shown = bytes; }  // what hipMemGetInfo calls the device's memory (0: the limit)
void fake_pin_limit(size_t bytes) { pin_limit = bytes; }
long fake_launches() { return launches; }
long fake_launches_of(const char* part) {  // of kernels whose mangled name contains part
    std::lock_guard<std::mutex> lock(mu);
    long n = 0;
    for (const auto& k : launched)
        if (k.first.find(part) != std::string::npos) n += k.second;
    return n;
}
long fake_streams() { return streams; }
long fake_pins() { return pins; }
long fake_copies() { return transfers_h2d + transfers_d2h; }
size_t fake_used() { return used; }
size_t fake_pinned() { return pinned_bytes; }

hipError_t hipMalloc(void** p, size_t n) { return get(device, used, limit, p, n); }
hipError_t hipFree(void* p) { return put(device, used, p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    const hipError_t e = get(pinned, pinned_bytes, pin_limit, p, n);
    pins += e == hipSuccess;
    return e;
}
hipError_t hipHostFree(void* p) { return put(pinned, pinned_bytes, p); }
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    std::lock_guard<std::mutex> lock(mu);
    *t = shown ? shown : limit;
    *f = *t > used ? *t - used : 0;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { return copy(d, s, n, k); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return copy(d, s, n, k); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) {
    *s = handle<hipStream_t>();
    streams++;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = handle<hipGraph_t>(), hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return *x = handle<hipGraphExec_t>(), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = handle<hipEvent_t>(), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = handle<hipEvent_t>(), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 163840;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* scratch = std::calloc(1, (size_t)8 << 20);
    return *p = scratch, hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { return *n = 2, hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "refused"; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    std::lock_guard<std::mutex> lock(mu);
    launched[kernels[f]]++;
    return launches++ == refuse ? fail(hipErrorLaunchFailure) : hipSuccess;
}
// what a launch expression and the registration of the kernels compile to
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    cfg_grid = g;
    cfg_block = b;
    cfg_lds = lds;
    cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = cfg_grid;
    *b = cfg_block;
    *lds = cfg_lds;
    *s = cfg_stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* module = nullptr;
    return &module;
}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}
