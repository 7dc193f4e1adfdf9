// A HIP runtime without a GPU, for tests of the library's host code: device
// memory is host memory, kernels are recorded by name and not run, an
// allocation can be made to fail (leaving its error behind, as HIP does, until
// hipGetLastError takes it), launches of 2^32 threads or more along a dimension
// are refused (HIP runs a part of them), and a stream under capture refuses
// allocations and synchronous copies.  Host allocations (operator new) can be
// made to fail too.  Loaded before the library under HIP's own soname.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>
#include <vector>

typedef int err_t;   // hipError_t
enum { ok = 0, invalid = 1, oom = 2, invalid_configuration = 9, capture_unsupported = 900 };
struct dim { unsigned x, y, z; };

namespace {
struct launch { std::string name; void* stream; unsigned grid; unsigned long long words[14]; };   // words: of its first argument
struct event { size_t at = 0; };
std::map<const void*, std::string> g_kernels;
std::vector<launch> g_launches;
std::map<std::string, float> g_cost;      // ms per launch, by part of the kernel's name
struct block { size_t bytes, number; };
std::map<void*, block> g_blocks;
std::vector<size_t> g_allocated;          // every allocation's bytes, in order
size_t g_fail_from = ~(size_t)0, g_fail_to = ~(size_t)0, g_bytes = 0;
size_t g_host_from = ~(size_t)0;
void* g_capturing = nullptr;              // the stream under capture
bool g_capture_broken = false;
err_t g_last = ok;
struct { dim grid, block; size_t lds; void* stream; } g_call;
err_t set(err_t e) { if (e != ok) g_last = e; return e; }
err_t uncapturable() { if (!g_capturing) return ok; g_capture_broken = true; return set(capture_unsupported); }
}  // namespace

void* operator new(size_t n)
{
    void* p = n >= g_host_from ? nullptr : std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" {
// ---- controls for the tests
void fake_fail_allocations(size_t from, size_t to) { g_fail_from = from; g_fail_to = to; }   // of from <= bytes < to
void fake_fail_host_allocations(size_t from) { g_host_from = from; }
int fake_allocations() { return (int)g_allocated.size(); }
size_t fake_allocated(int i) { return g_allocated[(size_t)i]; }
void fake_capture(void* stream) { g_capturing = stream; g_capture_broken = false; }
int fake_capture_broken() { return g_capture_broken; }
size_t fake_device_bytes() { return g_bytes; }
size_t fake_blocks() { return g_blocks.size(); }
size_t fake_block(size_t i)   // number of the i-th block in use, in the order of their allocation
{
    std::vector<size_t> n;
    for (const auto& b : g_blocks) n.push_back(b.second.number);
    std::sort(n.begin(), n.end());
    return n[i];
}
void fake_cost(const char* part, float ms) { g_cost[part] = ms; }
void fake_clear_launches() { g_launches.clear(); }
int fake_launches() { return (int)g_launches.size(); }
const char* fake_launch_name(int i) { return g_launches[(size_t)i].name.c_str(); }
void* fake_launch_stream(int i) { return g_launches[(size_t)i].stream; }
unsigned long long fake_launch_word(int i, int k) { return g_launches[(size_t)i].words[k]; }
unsigned fake_launch_grid(int i) { return g_launches[(size_t)i].grid; }

// ---- the runtime
void** __hipRegisterFatBinary(const void*) { static void* p; return &p; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim*, dim*, int*)
{
    g_kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
err_t __hipPushCallConfiguration(dim g, dim b, size_t lds, void* s) { g_call = {g, b, lds, s}; return ok; }
err_t __hipPopCallConfiguration(dim* g, dim* b, size_t* lds, void** s)
{
    *g = g_call.grid; *b = g_call.block; *lds = g_call.lds; *s = g_call.stream;
    return ok;
}
err_t hipLaunchKernel(const void* f, dim g, dim b, void** args, size_t, void* s)
{
    if ((size_t)g.x * b.x >> 32 || (size_t)g.y * b.y >> 32 || (size_t)g.z * b.z >> 32) return set(invalid_configuration);
    launch l{g_kernels[f], s, g.x, {}};
    std::memcpy(l.words, args[0], sizeof(l.words));
    g_launches.push_back(l);
    return ok;
}
err_t hipGetLastError() { const err_t e = g_last; g_last = ok; return e; }
const char* hipGetErrorString(err_t e) { return e == ok ? "no error" : e == oom ? "out of memory" : "error"; }
err_t hipGetDeviceCount(int* n) { *n = 1; return ok; }
err_t hipGetDevice(int* d) { *d = 0; return ok; }
err_t hipSetDevice(int d) { return d == 0 ? ok : set(invalid); }
err_t hipDeviceGetAttribute(int* v, int, int) { *v = 256; return ok; }
err_t hipDeviceSynchronize() { return uncapturable(); }
err_t hipDriverGetVersion(int* v) { *v = 0; return ok; }
err_t hipRuntimeGetVersion(int* v) { *v = 0; return ok; }
err_t hipGetDevicePropertiesR0600(void*, int) { return set(invalid); }
err_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)1 << 38; return ok; }
err_t hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (uncapturable() != ok) return capture_unsupported;
    g_allocated.push_back(n);
    if (n >= g_fail_from && n < g_fail_to) return set(oom);
    *p = std::malloc(n ? n : 1);
    if (!*p) return set(oom);
    g_blocks[*p] = {n, g_allocated.size()};
    g_bytes += n;
    return ok;
}
err_t hipFree(void* p)
{
    const auto it = g_blocks.find(p);
    if (it == g_blocks.end()) return p ? set(invalid) : ok;
    g_bytes -= it->second.bytes;
    g_blocks.erase(it);
    std::free(p);
    return ok;
}
err_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::malloc(n); return *p ? ok : set(oom); }
err_t hipHostFree(void* p) { std::free(p); return ok; }
err_t hipMemcpy(void* d, const void* s, size_t n, int)
{
    if (uncapturable() != ok) return capture_unsupported;
    std::memcpy(d, s, n);
    return ok;
}
err_t hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { std::memcpy(d, s, n); return ok; }
err_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, void*)
{
    for (size_t i = 0; i < h; ++i) std::memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
    return ok;
}
err_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return ok; }
err_t hipMemsetAsync(void* p, int v, size_t n, void*) { std::memset(p, v, n); return ok; }
err_t hipGetSymbolAddress(void** p, const void*) { static char block[1 << 20]; *p = block; return ok; }
err_t hipStreamCreate(void** s) { *s = std::malloc(1); return ok; }
err_t hipStreamCreateWithFlags(void** s, unsigned) { return hipStreamCreate(s); }
err_t hipStreamDestroy(void* s) { std::free(s); return ok; }
err_t hipStreamSynchronize(void*) { return uncapturable(); }
err_t hipStreamWaitEvent(void*, void*, unsigned) { return ok; }
err_t hipStreamIsCapturing(void* s, int* status)
{
    *status = s && s == g_capturing ? 1 : 0;
    return ok;
}
err_t hipStreamBeginCapture(void* s, int) { fake_capture(s); return ok; }
err_t hipStreamEndCapture(void*, void** g) { *g = std::malloc(1); g_capturing = nullptr; return g_capture_broken ? set(capture_unsupported) : ok; }
err_t hipGraphInstantiate(void** e, void*, void*, char*, size_t) { *e = std::malloc(1); return ok; }
err_t hipGraphLaunch(void*, void*) { return ok; }
err_t hipGraphDestroy(void* g) { std::free(g); return ok; }
err_t hipGraphExecDestroy(void* e) { std::free(e); return ok; }
err_t hipEventCreate(void** e) { *e = new event(); return ok; }
err_t hipEventCreateWithFlags(void** e, unsigned) { return hipEventCreate(e); }
err_t hipEventDestroy(void* e) { delete (event*)e; return ok; }
err_t hipEventRecord(void* e, void*) { ((event*)e)->at = g_launches.size(); return ok; }
err_t hipEventSynchronize(void*) { return ok; }
err_t hipEventElapsedTime(float* ms, void* a, void* b)
{
    *ms = 0.0f;
    for (size_t i = ((event*)a)->at; i < ((event*)b)->at; ++i) {
        float cost = 1.0f;
        for (const auto& c : g_cost)
            if (g_launches[i].name.find(c.first) != std::string::npos) cost = c.second;
        *ms += cost;
    }
    return ok;
}
}
