// A stand-in for the HIP runtime on the CPU: device memory is host memory,
// copies are copies, kernels do not run.  What the library asked for (kernel
// launches, allocations, blocking copies) is written down, and a call can be
// made to fail, so that tests without a GPU see the host's decisions.
// Loaded with global scope before libiss_hip.so, whose references bind here.
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

struct Dim3 {
    uint32_t x, y, z;
};
struct PointerAttribute {  // hipPointerAttribute_t
    int type, device;
    void *device_pointer, *host_pointer;
    int managed;
    unsigned flags;
};

namespace {
constexpr int kSuccess = 0, kInvalid = 1, kNoMemory = 2, kUnknown = 999;
std::mutex mu;
std::map<const void*, std::string> kernels;
struct Launch {
    std::string name;
    Dim3 grid, block;
};
std::vector<Launch> launches;
std::map<void*, size_t> live;
struct Call {
    Dim3 grid, block;
    size_t shared;
    void* stream;
};
thread_local std::vector<Call> calls;
int fail_device = 0, fail_host = 0;     // the n-th call from now that may fail does (0: none)
int64_t n_copies = 0, n_host = 0, largest = 0;
const char *known_begin = nullptr, *known_end = nullptr;
int known_type = 0;

bool fails(int* countdown) { return *countdown > 0 && --*countdown == 0; }
int allocate(void** p, size_t n, int* countdown) {
    std::lock_guard<std::mutex> g(mu);
    if (fails(countdown)) return kNoMemory;
    *p = std::calloc(1, n);
    live[*p] = n;
    if (static_cast<int64_t>(n) > largest) largest = static_cast<int64_t>(n);
    return kSuccess;
}
void release(void* p) {
    std::lock_guard<std::mutex> g(mu);
    live.erase(p);
    std::free(p);
}
}  // namespace

extern "C" {
// ---- what the tests read and set
void fake_reset() {
    std::lock_guard<std::mutex> g(mu);
    launches.clear();
    n_copies = n_host = largest = 0;
}
// the launches whose kernel name holds `part`; workgroups and threads of the last
int64_t fake_launched(const char* part, int64_t* groups, int64_t* threads) {
    std::lock_guard<std::mutex> g(mu);
    int64_t n = 0;
    *groups = *threads = -1;
    for (auto& l : launches)
        if (l.name.find(part) != std::string::npos) {
            n++;
            *groups = int64_t(l.grid.x) * l.grid.y * l.grid.z;
            *threads = int64_t(l.block.x) * l.block.y * l.block.z;
        }
    return n;
}
// the n-th device allocation, asynchronous copy or wait, and the n-th
// allocation of pinned memory
void fake_fail(int device_n, int host_n) {
    std::lock_guard<std::mutex> g(mu);
    fail_device = device_n;
    fail_host = host_n;
}
int64_t fake_copies() { return n_copies; }      // blocking copies
int64_t fake_host_allocs() { return n_host; }
int64_t fake_largest() { return largest; }      // bytes of the largest device allocation
void fake_known(const char* p, int64_t n, int type) {   // memory that the runtime knows (1 host, 2 device)
    known_begin = p;
    known_end = p + n;
    known_type = type;
}

// ---- the runtime
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
    calls.push_back({grid, block, shared, stream});
    return kSuccess;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
    const Call c = calls.back();
    calls.pop_back();
    *grid = c.grid;
    *block = c.block;
    *shared = c.shared;
    *stream = c.stream;
    return kSuccess;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void**, size_t, void*) {
    std::lock_guard<std::mutex> g(mu);
    launches.push_back({kernels[f], grid, block});
    return kSuccess;
}
int hipMalloc(void** p, size_t n) { return allocate(p, n, &fail_device); }
int hipFree(void* p) { release(p); return kSuccess; }
int hipHostMalloc(void** p, size_t n, unsigned) {
    n_host++;
    const int64_t before = largest;
    const int e = allocate(p, n, &fail_host);
    largest = before;
    return e;
}
int hipHostFree(void* p) { release(p); return kSuccess; }
int hipMemcpy(void* d, const void* s, size_t n, int) {
    n_copies++;
    std::memcpy(d, s, n);
    return kSuccess;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
    {
        std::lock_guard<std::mutex> g(mu);
        if (fails(&fail_device)) return kUnknown;
    }
    std::memcpy(d, s, n);
    return kSuccess;
}
int hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, int, void*) { return kSuccess; }
int hipMemsetAsync(void* p, int v, size_t n, void*) { std::memset(p, v, n); return kSuccess; }
int hipPointerGetAttributes(PointerAttribute* a, const void* p) {
    *a = PointerAttribute{};
    const char* c = static_cast<const char*>(p);
    if (c >= known_begin && c < known_end) a->type = known_type;
    return kSuccess;
}
int hipGetLastError() { return kSuccess; }
const char* hipGetErrorString(int) { return "error of the stand-in"; }
int hipGetDeviceCount(int* n) { *n = 1; return kSuccess; }
int hipGetDevicePropertiesR0600(void*, int) { return kUnknown; }
int hipSetDevice(int) { return kSuccess; }
int hipGetSymbolAddress(void** p, const void*) { *p = nullptr; return kInvalid; }
int hipFuncSetAttribute(const void*, int, int) { return kSuccess; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 1; return kSuccess; }
int hipStreamCreate(void** s) { *s = nullptr; return kSuccess; }
int hipStreamDestroy(void*) { return kSuccess; }
int hipStreamSynchronize(void*) {
    std::lock_guard<std::mutex> g(mu);
    return fails(&fail_device) ? kUnknown : kSuccess;
}
int hipStreamBeginCapture(void*, int) { return kSuccess; }
int hipStreamEndCapture(void*, void** graph) { *graph = nullptr; return kSuccess; }
int hipGraphInstantiate(void** exec, void*, void*, char*, size_t) { *exec = nullptr; return kSuccess; }
int hipGraphLaunch(void*, void*) { return kSuccess; }
int hipGraphDestroy(void*) { return kSuccess; }
int hipGraphExecDestroy(void*) { return kSuccess; }
int hipEventCreate(void** e) { *e = std::malloc(1); return kSuccess; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = std::malloc(1); return kSuccess; }
int hipEventDestroy(void* e) { std::free(e); return kSuccess; }
int hipEventRecord(void*, void*) { return kSuccess; }
int hipEventSynchronize(void*) { return kSuccess; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0.f; return kSuccess; }
}
