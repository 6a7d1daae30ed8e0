// hip_standin.cpp — a HIP runtime for tests of the library's host side without
// a GPU. Loaded with RTLD_GLOBAL ahead of libatv_hip.so, it takes the place of
// the calls that the library makes: device memory is host memory, copies are
// memcpy, and a kernel launch runs nothing. What it adds is what the tests ask:
// every allocation is known, the k-th one can be made to fail, freed blocks are
// never reused, and a launch or a replayed graph whose first argument points to
// a freed block is counted. (Kernels whose tables the host keeps take a table's
// address first.)
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <vector>

namespace {

constexpr int kOutOfMemory = 2, kSuccess = 0;
constexpr std::size_t kDeviceBytes = std::size_t(288) << 30;

struct Dim3 {
    std::uint32_t x, y, z;
};
struct Config {
    Dim3 grid, block;
    std::size_t shared;
    void* stream;
};
struct Graph {
    std::vector<const char*> first; // first argument of every launch, read as a pointer
};

std::map<const char*, std::size_t> live, dead;
std::size_t live_bytes = 0;
long fail_after = -1; // allocations until one fails (< 0: none does)
long stale = 0, launches = 0, captures = 0;
std::vector<Config> configs;
Graph* capturing = nullptr;

bool inside(const std::map<const char*, std::size_t>& m, const char* p) {
    auto it = m.upper_bound(p);
    if (it == m.begin())
        return false;
    --it;
    return p < it->first + it->second;
}

int allocate(void** out, std::size_t bytes, bool counted) {
    *out = nullptr;
    if (counted && fail_after >= 0 && fail_after-- == 0)
        return kOutOfMemory;
    if (bytes > kDeviceBytes || live_bytes + bytes > kDeviceBytes)
        return kOutOfMemory;
    void* p = std::calloc(bytes ? bytes : 1, 1);
    if (!p)
        return kOutOfMemory;
    if (counted) {
        live[static_cast<char*>(p)] = bytes;
        live_bytes += bytes;
    }
    *out = p;
    return kSuccess;
}

void launch(void** args) {
    const char* p = nullptr;
    std::memcpy(&p, args[0], sizeof(p));
    launches += 1;
    if (capturing)
        capturing->first.push_back(p);
    else if (inside(dead, p))
        stale += 1;
}

} // namespace

extern "C" {

// ---- what the tests ask ----
void standin_fail_after(long n) { fail_after = n; }
long standin_failures_left() { return fail_after; }
long standin_stale() { return stale; }
long standin_launches() { return launches; }
long standin_captures() { return captures; }
// sizes of the live allocations, ascending; returns their number
long standin_live(std::int64_t* sizes, long cap) {
    std::multiset<std::size_t> s;
    for (const auto& kv : live)
        s.insert(kv.second);
    long k = 0;
    for (std::size_t v : s)
        if (k < cap)
            sizes[k++] = static_cast<std::int64_t>(v);
    return static_cast<long>(s.size());
}

// ---- the runtime's calls ----
int hipSetDevice(int) { return kSuccess; }
int hipGetLastError() { return kSuccess; }
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "stand-in"; }
int hipMalloc(void** p, std::size_t bytes) { return allocate(p, bytes, true); }
int hipFree(void* p) {
    const auto it = live.find(static_cast<char*>(p));
    if (it == live.end())
        std::abort(); // freed twice, or never allocated
    live_bytes -= it->second;
    dead[it->first] = it->second;
    live.erase(it);
    return kSuccess;
}
int hipHostMalloc(void** p, std::size_t bytes, unsigned) { return allocate(p, bytes, false); }
int hipHostFree(void* p) {
    std::free(p);
    return kSuccess;
}
int hipMemcpy(void* d, const void* s, std::size_t n, int) {
    std::memcpy(d, s, n);
    return kSuccess;
}
int hipMemcpyAsync(void* d, const void* s, std::size_t n, int, void*) {
    std::memcpy(d, s, n);
    return kSuccess;
}
int hipMemset(void* d, int v, std::size_t n) {
    std::memset(d, v, n);
    return kSuccess;
}
int hipMemsetAsync(void* d, int v, std::size_t n, void*) {
    std::memset(d, v, n);
    return kSuccess;
}
int hipMemGetInfo(std::size_t* f, std::size_t* t) {
    *t = kDeviceBytes;
    *f = kDeviceBytes - live_bytes;
    return kSuccess;
}
int hipGetSymbolAddress(void** p, const void*) {
    static char block[1 << 20];
    *p = block;
    return kSuccess;
}
int hipStreamCreateWithFlags(void** s, unsigned) {
    static int tag;
    *s = &tag;
    return kSuccess;
}
int hipStreamDestroy(void*) { return kSuccess; }
int hipStreamSynchronize(void*) { return kSuccess; }
int hipEventCreate(void** e) {
    static int tag;
    *e = &tag;
    return kSuccess;
}
int hipEventDestroy(void*) { return kSuccess; }
int hipEventRecord(void*, void*) { return kSuccess; }
int hipEventSynchronize(void*) { return kSuccess; }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 1.0f;
    return kSuccess;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, std::size_t sh, void* st) {
    configs.push_back(Config{g, b, sh, st});
    return kSuccess;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, std::size_t* sh, void** st) {
    const Config c = configs.back();
    configs.pop_back();
    *g = c.grid;
    *b = c.block;
    *sh = c.shared;
    *st = c.stream;
    return kSuccess;
}
int hipLaunchKernel(const void*, Dim3, Dim3, void** args, std::size_t, void*) {
    launch(args);
    return kSuccess;
}
int hipExtLaunchKernel(const void*, Dim3, Dim3, void** args, std::size_t, void*, void*, void*, int) {
    launch(args);
    return kSuccess;
}
int hipStreamBeginCapture(void*, int) {
    capturing = new Graph();
    captures += 1;
    return kSuccess;
}
int hipStreamEndCapture(void*, void** g) {
    *g = capturing;
    capturing = nullptr;
    return kSuccess;
}
int hipGraphInstantiate(void** exec, void* g, void*, char*, std::size_t) {
    *exec = new Graph(*static_cast<Graph*>(g));
    return kSuccess;
}
int hipGraphDestroy(void* g) {
    delete static_cast<Graph*>(g);
    return kSuccess;
}
int hipGraphExecDestroy(void* e) {
    delete static_cast<Graph*>(e);
    return kSuccess;
}
int hipGraphLaunch(void* e, void*) {
    for (const char* p : static_cast<Graph*>(e)->first)
        if (inside(dead, p))
            stale += 1;
    return kSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, char*, int, std::size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}

} // extern "C"
