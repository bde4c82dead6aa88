// A host-only stand-in for the HIP runtime calls libspns.so makes: device memory
// is host memory, copies and fills run at once, kernels are only logged.  Two
// devices.  What a real runtime would refuse, or what would reach the wrong
// queue, is an error here: a kernel launch or an event on a stream of another
// device than the calling thread's current one.
// Loaded with RTLD_GLOBAL before libspns.so (tests/host_hip.py).
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include <malloc.h>

#include <hip/hip_runtime_api.h>

namespace {
std::mutex mu;
std::string text;                       // one line per operation that ran
std::map<const void*, std::string> names;
std::map<char*, size_t> blocks;  // device memory
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;
thread_local long fail_alloc = -1;      // the library's allocations until one throws; < 0: none does
thread_local bool inside = false;       // in a call below, whose own allocations do not count
struct Inside {
    Inside() { inside = true; }
    ~Inside() { inside = false; }
};
struct Stream { int dev; std::vector<std::string>* capture = nullptr; };
struct Event { int dev; };
Stream null_stream{0};

Stream* of(hipStream_t s) { return s ? (Stream*)s : &null_stream; }
void note(hipStream_t s, const std::string& line)
{
    std::lock_guard<std::mutex> lk(mu);
    if (of(s)->capture) of(s)->capture->push_back(line);
    else text += line + "\n";
}
// size of the device block that holds p, 0 for host memory
size_t block_of(const void* p)
{
    std::lock_guard<std::mutex> lk(mu);
    auto it = blocks.upper_bound((char*)p);
    if (it == blocks.begin()) return 0;
    --it;
    return (char*)p < it->first + it->second ? it->second : 0;
}
void count(const char* call) { const Inside in; note(nullptr, std::string("call ") + call); }
}  // namespace

void* operator new(size_t n)
{
    if (!inside && fail_alloc >= 0 && fail_alloc-- == 0) throw std::bad_alloc();
    void* p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
// freed objects are overwritten, so that a later use shows
void operator delete(void* p) noexcept
{
    if (p) std::memset(p, 0xdd, malloc_usable_size(p));
    asm volatile("" ::"r"(p) : "memory");  // or the fill is dropped as dead
    std::free(p);
}
void operator delete(void* p, size_t) noexcept { operator delete(p); }

extern "C" {
// for the tests
const char* host_hip_log() { return text.c_str(); }
void host_hip_clear() { text.clear(); }
void host_hip_fail_alloc(long after) { fail_alloc = after; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names[host] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t);
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*);
static thread_local struct { dim3 g, b; size_t shm; hipStream_t s; } cfg;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shm, hipStream_t s) { cfg = {g, b, shm, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shm, hipStream_t* s)
{
    *g = cfg.g; *b = cfg.b; *shm = cfg.shm; *s = cfg.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t s)
{
    if (of(s)->dev != current) return last = hipErrorInvalidHandle;
    const Inside in;
    note(s, "kernel " + names[f] + " " + std::to_string(g.x) + "x" + std::to_string(g.y) + " " + std::to_string(b.x));
    return hipSuccess;
}

hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d)
{
    if (d < 0 || d > 1) return hipErrorInvalidDevice;
    current = d;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { count("hipDeviceGetAttribute"); *v = 256; return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = size_t(1) << 33; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
    count("hipOccupancyMaxActiveBlocksPerMultiprocessor");
    *n = 2;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) { std::memset(a, 0, sizeof *a); return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = nullptr; return hipErrorInvalidSymbol; }
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }

hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(n ? n : 1, 1); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n)
{
    const hipError_t e = hipHostMalloc(p, n, 0);
    std::lock_guard<std::mutex> lk(mu);
    blocks[(char*)*p] = n;
    return e;
}
hipError_t hipFree(void* p)
{
    {
        std::lock_guard<std::mutex> lk(mu);
        blocks.erase((char*)p);
    }
    return hipHostFree(p);
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st)
{
    const Inside in;
    note(st, "copy " + std::to_string(n) + " to " + std::to_string(block_of(d)) + " from " + std::to_string(block_of(s)));
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t)
{
    for (size_t i = 0; i < h; i++) std::memcpy((char*)d + i * dp, (const char*)s + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t) new Stream{current}; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete (Stream*)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode)
{
    count("hipStreamBeginCapture");
    of(s)->capture = new std::vector<std::string>;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g)
{
    *g = (hipGraph_t)of(s)->capture;
    of(s)->capture = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t)
{
    *e = (hipGraphExec_t) new std::vector<std::string>(*(std::vector<std::string>*)g);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete (std::vector<std::string>*)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete (std::vector<std::string>*)e; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t s)
{
    for (const std::string& l : *(std::vector<std::string>*)e) note(s, l);
    return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t) new Event{current}; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Event*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return of(s)->dev == ((Event*)e)->dev ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
}
