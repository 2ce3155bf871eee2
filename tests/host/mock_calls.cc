// Test infrastructure: a CPU stand-in for the HIP calls of the library's host
// code (prk_api.hip, batch.hip, autotune.hip), for what a call asks of the
// runtime: on which device and with which grid it launches, which sweeps and
// passes it enqueues.  Kernels do not run.  There are two devices; every
// thread starts on device 0, as in HIP.  Device memory is reserve-only host
// memory that remembers its device.
#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "prk_internal.hpp"
#include "sweep.hpp"

using namespace prk;

namespace {
struct Alloc {
    size_t bytes;
    int device;
};
struct Kernel {
    unsigned grid, block;
    int device;
};
std::mutex g_mu;
std::map<const char *, Alloc> g_allocs;
std::vector<Kernel> g_kernels;
struct Sweeps {
    int sweeps, any, rows, wgs;
    long long reach;  // bytes from the grid's start to the end of what a row before the last loads
    const void *in, *in_next;
};
std::vector<Sweeps> g_sweeps;  // launch_sweep (sweeps = 1, any = -1) and launch_pass calls
thread_local int t_device = 0;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
thread_local std::vector<Config> t_config;
struct Stream {
    int device;
};

int record(const SweepPlan &p, int sweeps, int any, const void *in, const void *in_next)
{
    const unsigned row_bytes = (unsigned)(p.pitch * (long long)dtype_size(p.dtype));
    const unsigned load = p.mode == MODE_DWORD ? row_load_bytes<MODE_DWORD>(row_bytes, false) : row_bytes;
    std::lock_guard<std::mutex> l(g_mu);
    g_sweeps.push_back(Sweeps{sweeps, any, p.rows_per_wave, p.wgs_per_cu, (long long)(p.span.nrows - 2) * row_bytes + load,
                              in, in_next});
    return 0;
}
}  // namespace

namespace prk {
#define PRK_MOCK_DTYPE(d)                                                                                       \
    int launch_sweep_##d(const SweepPlan &p, const void *in, void *in_next, void *, hipStream_t)                \
    {                                                                                                           \
        return p.load_only ? 0 : record(p, 1, -1, in, in_next);                                                 \
    }                                                                                                           \
    int launch_pass_##d(const SweepPlan &p, int sweeps, bool any, const void *in, void *in_next, void *, hipStream_t) \
    {                                                                                                           \
        return sweeps ? record(p, sweeps, any, in, in_next) : 0;                                                \
    }
PRK_MOCK_DTYPE(f64)
PRK_MOCK_DTYPE(f32)
PRK_MOCK_DTYPE(bf16)
}  // namespace prk

extern "C" {
// What the tests read and set.
void mock_reset(void)
{
    std::lock_guard<std::mutex> l(g_mu);
    g_kernels.clear();
    g_sweeps.clear();
}
int mock_kernels(void) { return (int)g_kernels.size(); }
void mock_kernel(int i, unsigned *v)
{
    v[0] = g_kernels[i].grid;
    v[1] = g_kernels[i].block;
    v[2] = (unsigned)g_kernels[i].device;
}
int mock_sweeps(void) { return (int)g_sweeps.size(); }
void mock_sweep(int i, long long *v)
{
    const Sweeps &s = g_sweeps[i];
    const long long x[] = {s.sweeps, s.any, s.rows, s.wgs, s.reach, (long long)s.in, (long long)s.in_next};
    std::memcpy(v, x, sizeof x);
}
int mock_bytes_on(int device)  // MiB allocated there
{
    std::lock_guard<std::mutex> l(g_mu);
    size_t n = 0;
    for (auto &a : g_allocs)
        if (a.second.device == device) n += a.second.bytes;
    return (int)((n + (1u << 20) - 1) >> 20);
}

hipError_t hipGetDevice(int *d)
{
    *d = t_device;
    return hipSuccess;
}
hipError_t hipSetDevice(int d)
{
    if (d < 0 || d > 1) return hipErrorInvalidDevice;
    t_device = d;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n)
{
    void *m = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> l(g_mu);
    g_allocs[(const char *)m] = Alloc{n, t_device};
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    std::lock_guard<std::mutex> l(g_mu);
    auto it = g_allocs.find((const char *)p);
    if (it == g_allocs.end()) return hipErrorInvalidValue;
    munmap(p, it->second.bytes ? it->second.bytes : 1);
    g_allocs.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = std::calloc(1, n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned)
{
    *d = h;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind)
{
    for (size_t r = 0; r < h; ++r) std::memcpy((char *)d + r * dp, (const char *)s + r * sp, w);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = (hipStream_t) new Stream{t_device};
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) { return hipStreamCreateWithFlags(s, 0); }
hipError_t hipStreamDestroy(hipStream_t s)
{
    delete (Stream *)s;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = (hipEvent_t)std::calloc(1, 16);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    *g = (hipGraph_t)std::calloc(1, 16);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    *e = (hipGraphExec_t)std::calloc(1, 16);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e)
{
    std::free(e);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
    std::free(g);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
static thread_local hipError_t t_last = hipSuccess;
hipError_t hipGetLastError(void)
{
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipFuncGetAttributes(hipFuncAttributes *, const void *) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidSymbol; }

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    t_config.push_back(Config{grid, block, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s)
{
    const Config c = t_config.back();
    t_config.pop_back();
    *grid = c.grid;
    *block = c.block;
    *lds = c.lds;
    *s = c.stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, dim3 *, dim3 *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

// HIP refuses a grid of 2^32 threads or more in one dimension.
hipError_t hipLaunchKernel(const void *, dim3 grid, dim3 block, void **, size_t, hipStream_t s)
{
    if ((unsigned long long)grid.x * block.x >> 32 || !grid.x || !grid.y || !block.x)
        return t_last = hipErrorInvalidConfiguration;
    std::lock_guard<std::mutex> l(g_mu);
    g_kernels.push_back(Kernel{grid.x, block.x, s ? ((Stream *)s)->device : t_device});
    return hipSuccess;
}
}
