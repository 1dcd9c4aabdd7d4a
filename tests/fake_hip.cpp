// A stand-in for the HIP runtime, for CPU tests of the library's host code: loaded
// before the library with global symbols, its functions take the place of the
// runtime's. Device memory is host memory and kernels do not run, but are counted
// by name. Copies are queued and made when an event is found done. A "stuck" device
// finishes nothing, and the clock then runs ten seconds at each look, so that the
// library's bounded waits end at once.

#include <hip/hip_runtime_api.h>
#include <time.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

namespace {
std::vector<std::function<void()>> g_queue;
bool g_stuck = false;
int g_polls = 0, g_polls_left = 0;  // a wait finds its event done after this many looks
size_t g_malloc_fails = 0;          // device allocations of this many bytes fail
int g_copy_fails = -1;              // the copy of this number (from now, from 0) fails
int g_unbounded = 0;                // waits without a limit
std::map<void*, size_t> g_pinned;
std::map<const void*, std::string> g_names;
std::string g_launches;
long long g_skew_ns = 0;
hipError_t g_last = hipSuccess;

hipError_t ret(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}
void drain() {
    for (auto& f : g_queue) f();
    g_queue.clear();
}
}  // namespace

namespace std::chrono {
inline namespace _V2 {
steady_clock::time_point steady_clock::now() noexcept {
    timespec t;
    clock_gettime(CLOCK_MONOTONIC, &t);
    if (g_stuck) g_skew_ns += 10'000'000'000LL;
    return time_point(duration((long long)t.tv_sec * 1'000'000'000LL + t.tv_nsec + g_skew_ns));
}
}  // namespace _V2
}  // namespace std::chrono

extern "C" {
// controls of the tests
void fake_stuck(int on) { g_stuck = on != 0; }
void fake_polls(int n) { g_polls = g_polls_left = n; }
void fake_malloc_fails(size_t n) { g_malloc_fails = n; }
void fake_copy_fails(int n) { g_copy_fails = n; }
int fake_unbounded_waits() { return g_unbounded; }
size_t fake_pinned_bytes() {
    size_t n = 0;
    for (auto& p : g_pinned) n += p.second;
    return n;
}
const char* fake_launches() {  // the kernels launched since the last call, one to a line
    static std::string out;
    out.swap(g_launches);
    g_launches.clear();
    return out.c_str();
}

void** __hipRegisterFatBinary(const void*) {
    static void* h = nullptr;
    return &h;
}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    g_names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->name, "stand-in");
    std::strcpy(p->gcnArchName, "none");
    p->multiProcessorCount = 256;
    p->totalGlobalMem = (size_t)288 << 30;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetLastError() {
    hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) { return *p = const_cast<void*>(s), hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) {
    if (n == g_malloc_fails) return ret(hipErrorOutOfMemory);
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    g_pinned[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    if (g_stuck) g_unbounded++;  // the runtime's waits for the device
    g_pinned.erase(p);
    return std::free(p), hipSuccess;
}

hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind k, hipStream_t) {
    if (g_copy_fails >= 0 && g_copy_fails-- == 0) return hipErrorInvalidValue;
    auto pinned = [&](const void* p) {
        auto it = g_pinned.upper_bound(const_cast<void*>(p));
        if (it == g_pinned.begin()) return false;
        --it;
        return (const char*)p + n <= (const char*)it->first + it->second;
    };
    g_queue.push_back([=] { std::memcpy(dst, src, n); });
    // pageable memory: the call returns when the copy is made
    if ((k == hipMemcpyHostToDevice && !pinned(src)) || (k == hipMemcpyDeviceToHost && !pinned(dst))) {
        if (g_stuck)
            g_unbounded++;
        else
            drain();
    }
    return hipSuccess;
}

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = (hipEvent_t)std::malloc(1), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free((void*)e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return g_polls_left = g_polls, hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) {
    if (g_stuck || g_polls_left-- > 0) return hipErrorNotReady;
    drain();
    return hipSuccess;
}
static hipError_t unbounded() {
    if (g_stuck)
        g_unbounded++;
    else
        drain();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return unbounded(); }
hipError_t hipStreamSynchronize(hipStream_t) { return unbounded(); }
hipError_t hipDeviceSynchronize() { return unbounded(); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    return *s = hipStreamCaptureStatusNone, hipSuccess;
}

static hipError_t launched(const void* f) {
    auto it = g_names.find(f);
    g_launches += (it == g_names.end() ? std::string("?") : it->second) + "\n";
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) { return launched(f); }
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) {
    return launched(f);
}
static thread_local struct {
    dim3 g, b;
    size_t s;
    hipStream_t st;
} t_call;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
    t_call = {g, b, s, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
    *g = t_call.g, *b = t_call.b, *s = t_call.s, *st = t_call.st;
    return hipSuccess;
}
}
