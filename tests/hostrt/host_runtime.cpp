// host_runtime.cpp -- the HIP entry points that the library calls, on host
// memory and without kernels: the library's host code linked against it runs
// on the CPU, so that what it does on errors, on other devices and from
// several threads can be tested without a GPU.
//
//   - two devices; every thread has a current one (0 at first), streams and
//     events belong to the one they were made on, and recording an event on,
//     or launching on, another device's stream is refused as HIP refuses it;
//   - memory of both kinds is host memory and counted.  Device allocations are
//     whole pages, one after the other, so that neighbours touch; a copy that
//     does not lie within one is refused as HIP refuses it.  Copies are done
//     at once;
//   - a launch does nothing but report its kernel's name and arguments to the
//     test's callback (hr_on_launch), which may write what the kernel would;
//   - any entry point can be made to fail once (hr_fail), and so can the
//     library's own allocations on the calling thread (hr_fail_new).
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <thread>

namespace {

std::mutex g_mu;
std::map<std::string, long> g_calls;          // calls of every entry point
std::map<std::string, long> g_launches;       // launches of every kernel
std::map<const void *, std::string> g_names;  // kernels by host handle
std::string g_fail_name;
long g_fail_after = -1;
long g_delay_us = 0;  // of hipHostMalloc
void (*g_launch_cb)(const char *, void **) = nullptr;
thread_local int t_device = 0;
thread_local long t_new = -1;
thread_local hipError_t t_last = hipSuccess;
thread_local struct {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} t_cfg;

struct Obj {
    int device;
};

// the runtime's own allocations do not fail
struct NoFail {
    const long saved = t_new;
    NoFail() { t_new = -1; }
    ~NoFail() { t_new = saved; }
};

// device memory: pages of one reserved range, never handed out twice
constexpr size_t kPage = 4096, kRange = size_t(1) << 38;
char *g_base = nullptr, *g_next = nullptr;
std::map<char *, size_t> g_blocks;  // live allocations

// whether [p, p + n) is no device memory, or lies within one allocation
bool in_one_block(const void *p, size_t n)
{
    const NoFail nf;
    std::lock_guard<std::mutex> lk(g_mu);
    char *c = static_cast<char *>(const_cast<void *>(p));
    if (!g_base || c < g_base || c >= g_base + kRange) return true;
    auto it = g_blocks.upper_bound(c);
    if (it == g_blocks.begin()) return false;
    --it;
    return c + n <= it->first + it->second;
}

hipError_t enter(const char *name)
{
    const NoFail nf;
    std::lock_guard<std::mutex> lk(g_mu);
    ++g_calls[name];
    if (g_fail_after >= 0 && g_fail_name == name && g_fail_after-- == 0)
        return t_last = hipErrorOutOfMemory;
    return hipSuccess;
}

#define ENTER()                                        \
    do {                                               \
        const hipError_t e_ = enter(__func__);         \
        if (e_ != hipSuccess) return e_;               \
    } while (0)

template <class T>
T make()
{
    const NoFail nf;
    return reinterpret_cast<T>(new Obj{t_device});
}

template <class T>
int device_of(T t)
{
    return reinterpret_cast<Obj *>(t)->device;
}

void *allocate(size_t n)
{
    if (t_new >= 0 && t_new-- == 0) throw std::bad_alloc();
    void *p = std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}

}  // namespace

void *operator new(size_t n) { return allocate(n); }
void *operator new[](size_t n) { return allocate(n); }
void operator delete(void *p) noexcept { std::free(p); }
void operator delete[](void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
void operator delete[](void *p, size_t) noexcept { std::free(p); }

extern "C" {

// ----------------------------------------------------------- for tests --
// the (after + 1)-th allocation of this thread from now on fails; returns
// whether the one asked for last is still to come
int hr_fail_new(long after)
{
    const int waiting = t_new >= 0;
    t_new = after;
    return waiting;
}
long hr_calls(const char *name)
{
    std::lock_guard<std::mutex> lk(g_mu);
    return g_calls[name];
}
// launches of the kernels whose mangled name contains part
long hr_launches(const char *part)
{
    std::lock_guard<std::mutex> lk(g_mu);
    long n = 0;
    for (auto &q : g_launches)
        if (q.first.find(part) != std::string::npos) n += q.second;
    return n;
}
void hr_on_launch(void (*cb)(const char *, void **)) { g_launch_cb = cb; }
// the (after + 1)-th call of name from now on fails; after < 0: none
void hr_fail(const char *name, long after)
{
    std::lock_guard<std::mutex> lk(g_mu);
    g_fail_name = name;
    g_fail_after = after;
}
void hr_pin_delay_us(long us) { g_delay_us = us; }
void hr_set_device(int d) { t_device = d; }
int hr_device() { return t_device; }

// ------------------------------------------------------------- devices --
hipError_t hipGetDeviceCount(int *n)
{
    *n = 2;
    return hipSuccess;
}
hipError_t hipSetDevice(int d)
{
    ENTER();
    t_device = d;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    ENTER();
    *d = t_device;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->name, "host");
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 160 << 10;
    p->totalGlobalMem = size_t(1) << 38;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize()
{
    ENTER();
    return hipSuccess;
}
const char *hipGetErrorName(hipError_t e)
{
    return e == hipErrorOutOfMemory     ? "hipErrorOutOfMemory"
           : e == hipErrorInvalidHandle ? "hipErrorInvalidHandle"
           : e == hipErrorInvalidValue  ? "hipErrorInvalidValue"
                                        : "hipError";
}
hipError_t hipGetLastError()
{
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}

// -------------------------------------------------------------- memory --
hipError_t hipMalloc(void **p, size_t n)
{
    ENTER();
    const NoFail nf;
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_base) {
        void *m = mmap(nullptr, kRange, PROT_READ | PROT_WRITE,
                       MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        if (m == MAP_FAILED) return hipErrorOutOfMemory;
        g_base = g_next = static_cast<char *>(m);
    }
    const size_t b = (n + kPage - 1) / kPage * kPage;
    if (n == 0 || g_next + b > g_base + kRange) return hipErrorOutOfMemory;
    *p = g_next;
    g_blocks[g_next] = n;
    g_next += b;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    ENTER();
    const NoFail nf;
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_blocks.find(static_cast<char *>(p));
    if (it == g_blocks.end()) return p ? hipErrorInvalidValue : hipSuccess;
    madvise(p, (it->second + kPage - 1) / kPage * kPage, MADV_DONTNEED);
    g_blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    ENTER();
    if (g_delay_us) std::this_thread::sleep_for(std::chrono::microseconds(g_delay_us));
    *p = nullptr;
    return posix_memalign(p, 4096, n ? n : 1) == 0 ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p)
{
    ENTER();
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    ENTER();
    std::memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    ENTER();
    if (!in_one_block(d, n) || !in_one_block(s, n)) return hipErrorInvalidValue;
    std::memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    ENTER();
    if (!in_one_block(d, n)) return hipErrorInvalidValue;
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *)
{
    ENTER();
    std::memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *n, hipDeviceptr_t p)
{
    ENTER();
    *base = p;
    *n = size_t(1) << 40;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static char scratch[256];
    *p = scratch;
    return hipSuccess;
}

// --------------------------------------------------- streams and events --
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    ENTER();
    *s = make<hipStream_t>();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    ENTER();
    delete reinterpret_cast<Obj *>(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    ENTER();
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned)
{
    ENTER();
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    ENTER();
    *e = make<hipEvent_t>();
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    ENTER();
    delete reinterpret_cast<Obj *>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    ENTER();
    if (s && device_of(e) != device_of(s)) return t_last = hipErrorInvalidHandle;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t)
{
    ENTER();
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.f;
    return hipSuccess;
}

// ------------------------------------------------- graphs: none of them --
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

// ------------------------------------------------------------- kernels --
void **__hipRegisterFatBinary(const void *)
{
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, dim3 *, dim3 *, int *)
{
    std::lock_guard<std::mutex> lk(g_mu);
    g_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s)
{
    t_cfg = {grid, block, shared, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *s)
{
    *grid = t_cfg.grid;
    *block = t_cfg.block;
    *shared = t_cfg.shared;
    *s = t_cfg.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t s)
{
    ENTER();
    const NoFail nf;
    if (s && device_of(s) != t_device) return t_last = hipErrorInvalidHandle;
    if (grid.x == 0 || grid.y == 0 || grid.z == 0)
        return t_last = hipErrorInvalidConfiguration;
    std::string name;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        name = g_names[f];
        ++g_launches[name];
        if (g_fail_after >= 0 && name.find(g_fail_name) != std::string::npos &&
            g_fail_after-- == 0)
            return t_last = hipErrorOutOfMemory;
    }
    if (g_launch_cb) g_launch_cb(name.c_str(), args);
    return hipSuccess;
}

}  // extern "C"
