// A stand-in for the HIP runtime in host memory, for tests of the host code
// that prepares and launches kernels: device memory is ordinary memory with
// known extents, copies are checked against them, a kernel launch calls the
// test's function with the kernel's name and arguments and does nothing else.
// Loaded before libboxzy_hip.so with its symbols global (fakehip.py).
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {
std::mutex mu;
std::map<char *, size_t> dev;           // device allocations
std::map<const void *, std::string> kernels;
size_t pinned_limit = ~size_t(0), moved_limit = size_t(256) << 20;
long bad = 0;
bool no_new = false;  // operator new fails
typedef void (*launch_fn)(const char *name, const unsigned *grid, const unsigned *block, void **args);
launch_fn on_launch = nullptr;
struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local Config config;

// bytes from p to the end of its device allocation, or -1 for other memory
long room(const void *p)
{
    std::lock_guard<std::mutex> lk(mu);
    auto it = dev.upper_bound((char *)p);
    if (it == dev.begin()) return -1;
    --it;
    const long left = (long)(it->first + it->second - (const char *)p);
    return left >= 0 ? left : -1;
}
void check(const void *p, size_t n, const char *what)
{
    const long r = room(p);
    if (r < 0 || (size_t)r >= n) return;
    bad++;
    std::fprintf(stderr, "%s: %zu bytes where %ld are left\n", what, n, r);
}
}  // namespace

// the library's allocations (libstdc++'s own are malloc too)
void *operator new(size_t n)
{
    void *p = no_new ? nullptr : std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {

void fake_set(launch_fn f, size_t pinned) { on_launch = f, pinned_limit = pinned; }
long fake_room(const void *p) { return room(p); }
long fake_bad() { return bad; }
void fake_no_new(int on) { no_new = on != 0; }

hipError_t hipMalloc(void **p, size_t n)
{
    void *m = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> lk(mu);
    dev[(char *)m] = n;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> lk(mu);
    auto it = dev.find((char *)p);
    if (it == dev.end()) return hipSuccess;
    munmap(p, it->second ? it->second : 1);
    dev.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (n > pinned_limit) return hipErrorOutOfMemory;
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    check(d, n, "copy to");
    check(s, n, "copy from");
    if (n <= moved_limit && !bad) std::memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void *p, int, size_t n) { return check(p, n, "set"), hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { return *f = *t = size_t(288) << 30, hipSuccess; }

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t, hipStream_t)
{
    const unsigned g[3] = {grid.x, grid.y, grid.z}, b[3] = {block.x, block.y, block.z};
    if (g[0] == 0 || g[1] == 0 || g[2] == 0 || g[1] > 65535u || g[2] > 65535u) return hipErrorInvalidConfiguration;
    if (on_launch) on_launch(kernels[f].c_str(), g, b, args);
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t q) { return config = {g, b, s, q}, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *q)
{
    *g = config.grid, *b = config.block, *s = config.shared, *q = config.stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { return new void *[1](); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake HIP error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidSymbol; }

static int handle;
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)&handle, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return *g = (hipGraph_t)&handle, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)&handle, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { return *t = 0.f, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return *x = (hipGraphExec_t)&handle, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
}
