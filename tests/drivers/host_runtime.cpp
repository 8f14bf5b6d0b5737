// A HIP runtime on the host for tests of the library's host paths: memory is
// host memory, copies are copies, and a kernel launch only notes the kernel's
// name.  Loaded (RTLD_GLOBAL) before libgpe_hip.so it takes the runtime's
// place, so route choices, allocations and error paths run without a GPU.
// Signatures follow the public HIP API; types are opaque here.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct Dim3 {
    uint32_t x, y, z;
};

std::mutex mu;
std::map<const void*, std::string> kernels;          // host stub -> device name
std::map<void*, size_t> blocks;                      // live device allocations
std::string launches;                                // names of the launches since hh_reset, one a line
std::vector<std::pair<std::string, double>> costs;   // launch cost in ms of kernels whose name holds the text
double now_ms = 0.0;
size_t used = 0, total = (size_t)8 << 30;
int cus = 256;
long fail_malloc = 0, fail_upload = 0;               // countdown to a failing call, 0: none
long uploaded = 0;                                   // bytes copied from host memory since hh_reset
bool capturing = false;
Dim3 grid, block;
size_t shmem;
void* stream_arg;

constexpr int kOk = 0, kOutOfMemory = 2, kUnknown = 999;

int alloc(void** p, size_t n) {
    std::lock_guard<std::mutex> g(mu);
    if (fail_malloc > 0 && --fail_malloc == 0) return kOutOfMemory;
    if (used + n > total) return kOutOfMemory;
    *p = std::calloc(n ? n : 1, 1);
    if (!*p) return kOutOfMemory;
    blocks[*p] = n;
    used += n;
    return kOk;
}

int copy(void* d, const void* s, size_t n, int kind) {
    std::lock_guard<std::mutex> g(mu);
    if (kind == 1) {  // host to device
        if (fail_upload > 0 && --fail_upload == 0) return kUnknown;
        uploaded += (long)n;
    }
    std::memcpy(d, s, n);
    return kOk;
}

}  // namespace

extern "C" {

// ---- what a test sets and reads
void hh_reset() {
    launches.clear();
    uploaded = 0;
}
const char* hh_launches() { return launches.c_str(); }
long hh_uploaded() { return uploaded; }
void hh_fail(long nth_malloc, long nth_upload) {
    fail_malloc = nth_malloc;
    fail_upload = nth_upload;
}
void hh_memory(size_t bytes) { total = bytes; }
size_t hh_used() { return used; }
size_t hh_blocks() { return blocks.size(); }
void hh_cus(int n) { cus = n; }
void hh_capture(int on) { capturing = on != 0; }
void hh_cost(const char* text, double ms) { costs.emplace_back(text, ms); }

// ---- the runtime
void** __hipRegisterFatBinary(const void*) {
    static void* module[1];
    return module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
    kernels[stub] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void* s) {
    grid = g;
    block = b;
    shmem = sh;
    stream_arg = s;
    return kOk;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* sh, void** s) {
    *g = grid;
    *b = block;
    *sh = shmem;
    *s = stream_arg;
    return kOk;
}
int hipLaunchKernel(const void* stub, Dim3, Dim3, void**, size_t, void*) {
    std::lock_guard<std::mutex> g(mu);
    const std::string& name = kernels[stub];
    launches += name + "\n";
    double ms = 0.01;
    for (const auto& c : costs)
        if (name.find(c.first) != std::string::npos) ms = c.second;
    now_ms += ms;
    return kOk;
}
int hipMalloc(void** p, size_t n) { return alloc(p, n); }
int hipFree(void* p) {
    std::lock_guard<std::mutex> g(mu);
    auto it = blocks.find(p);
    if (it == blocks.end()) return p ? kUnknown : kOk;
    used -= it->second;
    blocks.erase(it);
    std::free(p);
    return kOk;
}
int hipMemGetInfo(size_t* f, size_t* t) {
    *f = total - used;
    *t = total;
    return kOk;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    return *p ? kOk : kOutOfMemory;
}
int hipHostFree(void* p) {
    std::free(p);
    return kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind) { return copy(d, s, n, kind); }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) { return copy(d, s, n, kind); }
int hipMemset(void* d, int v, size_t n) {
    std::memset(d, v, n);
    return kOk;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { return hipMemset(d, v, n); }
int hipGetDevice(int* d) {
    *d = 0;
    return kOk;
}
int hipSetDevice(int) { return kOk; }
int hipDeviceGetAttribute(int* v, int, int) {
    *v = cus;
    return kOk;
}
int hipGetLastError() { return kOk; }
const char* hipGetErrorString(int) { return "host runtime"; }
int hipGetSymbolAddress(void** p, const void*) {
    static char area[1 << 20];
    *p = area;
    return kOk;
}
int hipStreamCreateWithFlags(void** s, unsigned) {
    static char name;
    *s = &name;
    return kOk;
}
int hipStreamDestroy(void*) { return kOk; }
int hipStreamSynchronize(void*) { return kOk; }
int hipStreamWaitEvent(void*, void*, unsigned) { return kOk; }
int hipStreamIsCapturing(void*, int* status) {
    *status = capturing ? 1 : 0;
    return kOk;
}
int hipStreamBeginCapture(void*, int) { return kUnknown; }
int hipStreamEndCapture(void*, void**) { return kUnknown; }
int hipGraphInstantiate(void**, void*, void**, char*, size_t) { return kUnknown; }
int hipGraphLaunch(void*, void*) { return kUnknown; }
int hipGraphDestroy(void*) { return kOk; }
int hipGraphExecDestroy(void*) { return kOk; }
int hipEventCreate(void** e) {
    *e = new double(0.0);
    return kOk;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void* e) {
    delete (double*)e;
    return kOk;
}
int hipEventRecord(void* e, void*) {
    *(double*)e = now_ms;
    return kOk;
}
int hipEventSynchronize(void*) { return kOk; }
int hipEventElapsedTime(float* ms, void* a, void* b) {
    *ms = (float)(*(double*)b - *(double*)a);
    return kOk;
}
}
