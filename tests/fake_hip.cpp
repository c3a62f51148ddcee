// A HIP runtime on host memory for tests of the library's host code without a
// GPU: it defines the runtime entry points that libpa_admm.so calls, and loaded
// before that library (RTLD_GLOBAL) it takes their place.  Device memory is
// zeroed host memory, copies are memcpy (null operands are an error), kernels
// do nothing but are counted by name, and a chosen allocation fails.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
constexpr int OK = 0, INVALID = 1, OUT_OF_MEMORY = 2;
std::map<void*, size_t> mem;
std::map<const void*, std::string> names; // kernels by their host stub
std::map<std::string, long> launches;
std::map<const void*, std::string> vars;
std::map<std::string, size_t> var_bytes;
std::map<const void*, void*> var_mem;
long allocs = 0, fail_at = 0;
size_t live = 0;
long handles = 0; // streams, events and pinned allocations that are alive
uint32_t* last_pinned = nullptr;
char token; // handles: any address that is not null
struct Dim3 {
    uint32_t x, y, z;
};
} // namespace

extern "C" {
// ---- controls ----
void fake_fail_at(long nth) { // the nth allocation from now fails (0: none)
    fail_at = nth > 0 ? allocs + nth : 0;
}
long fake_allocs() { return allocs; }
size_t fake_live() { return live; }
long fake_handles() { return handles; }
long fake_launches(const char* part) { // of the kernels whose mangled name holds `part`
    long n = 0;
    for (auto& l : launches)
        if (l.first.find(part) != std::string::npos) n += l.second;
    return n;
}
size_t fake_var_bytes(const char* part) { // of the device variables whose name holds `part`
    size_t n = 0;
    for (auto& v : var_bytes)
        if (v.first.find(part) != std::string::npos) n += v.second;
    return n;
}
uint32_t* fake_last_pinned() { return last_pinned; }

// ---- memory ----
int hipMalloc(void** p, size_t bytes) {
    if (++allocs == fail_at) return OUT_OF_MEMORY;
    *p = std::calloc(bytes ? bytes : 1, 1);
    if (!*p) return OUT_OF_MEMORY;
    mem[*p] = bytes;
    live += bytes;
    return OK;
}
int hipFree(void* p) {
    auto it = mem.find(p);
    if (it == mem.end()) return p ? INVALID : OK;
    live -= it->second;
    mem.erase(it);
    std::free(p);
    return OK;
}
int hipHostMalloc(void** p, size_t bytes, unsigned) {
    *p = std::calloc(bytes, 1);
    last_pinned = static_cast<uint32_t*>(*p);
    handles++;
    return *p ? OK : OUT_OF_MEMORY;
}
int hipHostFree(void* p) {
    handles--;
    std::free(p);
    return OK;
}
int hipMemcpyAsync(void* d, const void* s, size_t bytes, int, void*) {
    if (bytes && (!d || !s)) return INVALID;
    if (bytes) std::memcpy(d, s, bytes);
    return OK;
}
int hipMemsetAsync(void* d, int v, size_t bytes, void*) {
    if (bytes && !d) return INVALID;
    if (bytes) std::memset(d, v, bytes);
    return OK;
}
int hipGetSymbolAddress(void** p, const void* symbol) {
    auto it = vars.find(symbol);
    if (it == vars.end()) return INVALID;
    void*& m = var_mem[symbol];
    if (!m) m = std::calloc(var_bytes[it->second], 1);
    *p = m;
    return OK;
}

// ---- modules and launches ----
void** __hipRegisterFatBinary(const void*) {
    static void* handle = &token;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names[stub] = name; }
void __hipRegisterVar(void**, void* var, char*, const char* name, int, size_t bytes, int, int) {
    vars[var] = name;
    var_bytes[name] = bytes;
}
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void*) { return OK; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* shared, void** stream) {
    *g = *b = Dim3{1, 1, 1};
    *shared = 0;
    *stream = nullptr;
    return OK;
}
int hipLaunchKernel(const void* stub, Dim3, Dim3, void**, size_t, void*) {
    launches[names[stub]]++;
    return OK;
}

// ---- devices, streams, events, graphs ----
int hipGetDeviceCount(int* n) {
    *n = 1;
    return OK;
}
int hipSetDevice(int) { return OK; }
int hipGetDevice(int* d) {
    *d = 0;
    return OK;
}
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 0;
    return OK;
}
int hipGetLastError() { return OK; }
const char* hipGetErrorString(int) { return "fake HIP error"; }
int hipStreamCreateWithFlags(void** s, unsigned) {
    *s = &token;
    handles++;
    return OK;
}
int hipStreamDestroy(void*) {
    handles--;
    return OK;
}
int hipStreamSynchronize(void*) { return OK; }
int hipStreamWaitEvent(void*, void*, unsigned) { return OK; }
int hipStreamBeginCapture(void*, int) { return OK; }
int hipStreamEndCapture(void*, void** g) {
    *g = &token;
    return OK;
}
int hipEventCreate(void** e) {
    *e = &token;
    handles++;
    return OK;
}
int hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void*) {
    handles--;
    return OK;
}
int hipEventRecord(void*, void*) { return OK; }
int hipEventSynchronize(void*) { return OK; }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 0.f;
    return OK;
}
int hipGraphInstantiate(void** e, void*, void**, char*, size_t) {
    *e = &token;
    return OK;
}
int hipGraphLaunch(void*, void*) { return OK; }
int hipGraphDestroy(void*) { return OK; }
int hipGraphExecDestroy(void*) { return OK; }
}
