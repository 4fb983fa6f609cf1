// A HIP runtime for the host side of the library alone, loaded before it: memory on the host,
// kernels that do nothing, and the order of the streams' work kept as vector clocks.  A test sees
// what a call leaves behind on its streams without a GPU.
//   stub_fail_copies(n)  the n-th hipMemcpyAsync from now on fails (0: none)
//   stub_busy()          launches the host has not waited for, over all streams
//   stub_bytes()         device memory asked for so far
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>

namespace {
using Clock = std::map<void*, long long>;  // stream -> launches on it
struct dim3 {
    uint32_t x, y, z;
};
Clock done;                       // launches the host has waited for
std::map<void*, Clock> streams;   // what each stream's next launch comes after
std::map<void*, Clock> events;    // what each event marks
struct Config {
    dim3 grid, block;
    size_t lds;
    void* stream;
} config;
int fail_in = 0;
long long asked = 0;
constexpr int kError = 999;  // hipErrorUnknown

void join(Clock& a, const Clock& b) {
    for (auto& t : b)
        if (a[t.first] < t.second) a[t.first] = t.second;
}
int alloc(void** p, size_t n) { return (*p = std::calloc(n ? n : 1, 1)) ? 0 : 2; }
void* handle() { return std::calloc(1, 8); }
}  // namespace

extern "C" {
void stub_fail_copies(int n) { fail_in = n; }
long long stub_bytes() { return asked; }
long long stub_busy() {
    long long n = 0;
    for (auto& s : streams) n += s.second[s.first] - done[s.first];
    return n;
}

void** __hipRegisterFatBinary(const void*) { return (void**)handle(); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, dim3*, dim3*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* s) {
    config = {g, b, lds, s};
    return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s) {
    *g = config.grid, *b = config.block, *lds = config.lds, *s = config.stream;
    return 0;
}
int hipLaunchKernel(const void*, dim3, dim3, void**, size_t, void* s) {
    ++streams[s][s];
    return 0;
}

int hipStreamCreate(void** s) { return (*s = handle()) ? 0 : 2; }
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void* s) {
    join(done, streams[s]);
    return 0;
}
int hipStreamWaitEvent(void* s, void* e, unsigned) {
    join(streams[s], events[e]);
    return 0;
}
int hipStreamBeginCapture(void*, int) { return kError; }
int hipStreamEndCapture(void*, void**) { return kError; }
int hipGraphInstantiate(void**, void*, void*, char*, size_t) { return kError; }
int hipGraphLaunch(void*, void*) { return kError; }
int hipGraphDestroy(void*) { return 0; }
int hipGraphExecDestroy(void*) { return 0; }

int hipEventCreate(void** e) { return (*e = handle()) ? 0 : 2; }
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void* e, void* s) {
    events[e] = streams[s];
    return 0;
}
int hipEventSynchronize(void* e) {
    join(done, events[e]);
    return 0;
}
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 0;
    return 0;
}

int hipMalloc(void** p, size_t n) {
    asked += (long long)n;
    return alloc(p, n);
}
int hipFree(void* p) {
    std::free(p);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return alloc(p, n); }
int hipHostFree(void* p) { return hipFree(p); }
int hipHostGetDevicePointer(void** d, void* h, unsigned) {
    *d = h;
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
    std::memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
    if (fail_in > 0 && --fail_in == 0) return kError;
    std::memcpy(d, s, n);
    return 0;
}
int hipMemset(void* d, int v, size_t n) {
    std::memset(d, v, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { return hipMemset(d, v, n); }
int hipGetSymbolAddress(void** p, const void*) { return alloc(p, (size_t)32 << 20); }

int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipGetDeviceCount(int* n) {
    *n = 1;
    return 0;
}
int hipGetDevicePropertiesR0600(void*, int) { return kError; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "stub"; }
}
