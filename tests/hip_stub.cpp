// A stand-in for the HIP runtime on a machine without a GPU: device memory is
// host memory, kernels are logged and not run.  Loaded with RTLD_GLOBAL before
// libmhx.so, its symbols take the place of the runtime's, so that the library's
// host code (allocation, errors, order of calls) can be tested through the C ABI.
//
// stub_fail(n) makes the n-th following call fail that can fail for want of a
// resource (allocations, copies, fills, launches, waits); errors stay until
// hipGetLastError takes them, as the runtime's do.  stub_log() is one line per
// call: malloc PTR BYTES, free PTR, memset PTR BYTES, memcpy DST BYTES, launch NAME
// and the pointers of `shown` kernels, attribute DEVICE NAME BYTES, destroy KIND,
// sync.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<char *, size_t> live;
std::map<const void *, std::string> names;
std::string logtext;
long fail_at = 0;
hipError_t last = hipSuccess;
int device = 0;
// kernels whose pointer arguments first .. last are logged: the table kernels'
// outputs, the tables read by the axisymmetric kernel
struct Shown {
    const char *kernel;
    int first, last;
};
const Shown shown[] = {{"k_plm_tables", 10, 13}, {"k_p_tables", 8, 11}, {"k_crec64", 3, 3}, {"k_axi", 2, 3}};
struct Config {
    dim3 grid, block;
    size_t shm;
    hipStream_t s;
} config;

void line(const char *what, const void *p, size_t n)
{
    char b[96];
    std::snprintf(b, sizeof(b), "%s %lx %zu\n", what, (unsigned long)(size_t)p, n);
    logtext += b;
}
hipError_t err(hipError_t e) { return last = e; }
bool failing() { return fail_at > 0 && --fail_at == 0; }
template <class T> hipError_t make(T *out)
{
    *out = reinterpret_cast<T>(std::malloc(1));
    return hipSuccess;
}
template <class T> hipError_t destroy(const char *kind, T h)
{
    logtext += std::string("destroy ") + kind + "\n";
    std::free(reinterpret_cast<void *>(h));
    return hipSuccess;
}
}  // namespace

extern "C" {

void stub_fail(long n) { fail_at = n; }
void stub_device(int d) { device = d; }
const char *stub_log() { return logtext.c_str(); }
void stub_clear() { logtext.clear(); }
size_t stub_live() { return live.size(); }
size_t stub_bytes()
{
    size_t n = 0;
    for (auto &e : live) n += e.second;
    return n;
}

hipError_t hipMalloc(void **p, size_t n)
{
    if (failing()) return err(hipErrorOutOfMemory);
    *p = std::malloc(n ? n : 1);
    live[static_cast<char *>(*p)] = n;
    line("malloc", *p, n);
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    line("free", p, 0);
    if (p && !live.erase(static_cast<char *>(p))) return err(hipErrorInvalidValue);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (failing()) return err(hipErrorOutOfMemory);
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n)
{
    if (failing()) return err(hipErrorUnknown);
    line("memset", p, n);
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    if (failing()) return err(hipErrorUnknown);
    line("memcpy", d, n);
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    auto it = live.upper_bound(const_cast<char *>(static_cast<const char *>(p)));
    if (it == live.begin()) return err(hipErrorInvalidValue);
    --it;
    if (static_cast<const char *>(p) >= it->first + it->second) return err(hipErrorInvalidValue);
    std::memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize()
{
    if (failing()) return err(hipErrorUnknown);
    logtext += "sync\n";
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = device;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int v)
{
    char b[32];
    std::snprintf(b, sizeof(b), " %d\n", v);
    logtext += "attribute " + std::to_string(device) + " " + names[f] + b;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s)
{
    *p = const_cast<void *>(s);
    return hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t *s) { return make(s); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return make(s); }
hipError_t hipStreamDestroy(hipStream_t s) { return destroy("stream", s); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return make(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return make(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return destroy("event", e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return make(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) { return make(x); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return destroy("graph", g); }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return destroy("exec", x); }

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shm, hipStream_t s)
{
    config = Config{grid, block, shm, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shm, hipStream_t *s)
{
    *grid = config.grid;
    *block = config.block;
    *shm = config.shm;
    *s = config.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t)
{
    if (failing()) return err(hipErrorLaunchFailure);
    const std::string &n = names[f];
    logtext += "launch " + n;
    for (const Shown &k : shown)
        if (n.find(k.kernel) != n.npos)
            for (int i = k.first; i <= k.last; ++i) {
                char b[24];
                std::snprintf(b, sizeof(b), " %lx", *static_cast<unsigned long *>(args[i]));
                logtext += b;
            }
    logtext += "\n";
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { return static_cast<void **>(std::calloc(1, sizeof(void *))); }
void __hipUnregisterFatBinary(void **h) { std::free(h); }
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

}  // extern "C"
