/*
 * A HIP runtime without a device, for CPU tests of the library's host path.
 *
 * Loaded with RTLD_GLOBAL before libslimtracin.so, it answers that library's
 * HIP calls: device and page-locked memory are host memory, copies are done
 * at once, kernels do not run. Every call is handed to a hook (fake_hook) by
 * name, with a kernel's mangled name and its arguments for a launch, so that
 * a test sees what the library queues, in which order, and can act in
 * between. fake_fail makes a coming call fail; fake_new_fail makes an
 * allocation of the library's C++ code throw.
 */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <map>
#include <mutex>
#include <new>
#include <string>

typedef int hipError_t;   /* 0: success */
struct dim3_ {
    uint32_t x, y, z;
};

static void (*g_hook)(const char *call, void **args) = nullptr;
static std::string g_fail_name;
static std::atomic<int> g_fail_in(0), g_new_in(0);
static std::mutex g_mu;
static std::map<const void *, std::string> g_kernels;
static std::map<uintptr_t, size_t> g_device, g_host;

/* allocations of this file are not the library's */
static thread_local int t_own;
struct Own {
    Own() { t_own++; }
    ~Own() { t_own--; }
};

static hipError_t call(const char *name, void **args = nullptr) {
    if (g_hook) g_hook(name, args);
    if (g_fail_in > 0 && g_fail_name == name && --g_fail_in == 0) return 999;
    return 0;
}
static hipError_t take(std::map<uintptr_t, size_t> &m, void **p, size_t n) {
    *p = calloc(1, n ? n : 1);
    if (!*p) return 2;
    Own own;
    std::lock_guard<std::mutex> lk(g_mu);
    m[(uintptr_t)*p] = n;
    return 0;
}
static void give(std::map<uintptr_t, size_t> &m, void *p) {
    if (!p) return;
    std::lock_guard<std::mutex> lk(g_mu);
    m.erase((uintptr_t)p);
    free(p);
}
static bool within(const std::map<uintptr_t, size_t> &m, const void *p) {
    auto it = m.upper_bound((uintptr_t)p);
    if (it == m.begin()) return false;
    --it;
    return (uintptr_t)p < it->first + it->second;
}

/* the library's own allocations (it finds this operator before libstdc++'s) */
void *operator new(size_t n) {
    if (!t_own && g_new_in > 0 && --g_new_in == 0) throw std::bad_alloc();
    void *p = malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}

extern "C" {

void fake_hook(void (*hook)(const char *, void **)) { g_hook = hook; }
void fake_fail(const char *name, int nth) {
    g_fail_name = name;
    g_fail_in = nth;
}
void fake_new_fail(int nth) { g_new_in = nth; }
int fake_new_left(void) { return g_new_in; }
/* page-locked memory of somebody else than the library */
void *fake_host_alloc(size_t n) {
    void *p = nullptr;
    return take(g_host, &p, n) ? nullptr : p;
}
size_t fake_device_bytes(void) {
    std::lock_guard<std::mutex> lk(g_mu);
    size_t n = 0;
    for (auto &kv : g_device) n += kv.second;
    return n;
}

void **__hipRegisterFatBinary(const void *) {
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
    g_kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

static thread_local struct {
    dim3_ grid, block;
    size_t lds;
    void *stream;
} t_config;
hipError_t __hipPushCallConfiguration(dim3_ grid, dim3_ block, size_t lds, void *stream) {
    t_config = {grid, block, lds, stream};
    return 0;
}
hipError_t __hipPopCallConfiguration(dim3_ *grid, dim3_ *block, size_t *lds, void **stream) {
    *grid = t_config.grid;
    *block = t_config.block;
    *lds = t_config.lds;
    *stream = t_config.stream;
    return 0;
}
hipError_t hipLaunchKernel(const void *f, dim3_, dim3_, void **args, size_t, void *) {
    std::string name;
    {
        Own own;
        name = "launch " + g_kernels[f];
    }
    return call(name.c_str(), args);
}

hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return 0;
}
hipError_t hipSetDevice(int) { return 0; }
hipError_t hipGetDevicePropertiesR0600(void *, int) { return 1; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *scratch = calloc(1, 256u << 20);
    *p = scratch;
    return 0;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 1;
    return call("hipOccupancyMaxActiveBlocksPerMultiprocessor");
}
hipError_t hipGetLastError(void) { return call("hipGetLastError"); }
const char *hipGetErrorString(hipError_t) { return "made to fail"; }

hipError_t hipMalloc(void **p, size_t n) {
    const hipError_t e = call("hipMalloc");
    return e ? e : take(g_device, p, n);
}
hipError_t hipFree(void *p) {
    give(g_device, p);
    return call("hipFree");
}
hipError_t hipMemGetInfo(size_t *free_b, size_t *total) {
    *free_b = *total = (size_t)288 << 30;
    return 0;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    const hipError_t e = call("hipHostMalloc");
    return e ? e : take(g_host, p, n);
}
hipError_t hipHostFree(void *p) {
    give(g_host, p);
    return call("hipHostFree");
}
hipError_t hipHostGetDevicePointer(void **d, void *p, unsigned) {
    *d = p;
    return 0;
}
hipError_t hipPointerGetAttributes(void *attr, const void *p) {
    struct {
        int type, device;
        void *device_pointer, *host_pointer;
        int managed;
        unsigned flags;
    } a = {0, 0, nullptr, nullptr, 0, 0};
    {
        std::lock_guard<std::mutex> lk(g_mu);
        a.type = within(g_host, p) ? 1 : within(g_device, p) ? 2 : 0;   /* host, device, unregistered */
    }
    memcpy(attr, &a, sizeof a);
    return call("hipPointerGetAttributes");
}
hipError_t hipMemset(void *p, int v, size_t n) {
    memset(p, v, n);
    return call("hipMemset");
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, int) {
    memmove(d, s, n);
    return call("hipMemcpy");
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) {
    void *args[3] = {d, (void *)s, (void *)n};
    const hipError_t e = call("hipMemcpyAsync", args);
    if (!e) memmove(d, s, n);
    return e;
}

hipError_t hipStreamCreateWithFlags(void **s, unsigned) {
    *s = malloc(1);
    return 0;
}
hipError_t hipStreamDestroy(void *s) {
    free(s);
    return 0;
}
hipError_t hipStreamSynchronize(void *) { return call("hipStreamSynchronize"); }
hipError_t hipStreamBeginCapture(void *, int) { return call("hipStreamBeginCapture"); }
hipError_t hipStreamEndCapture(void *, void **g) {
    *g = malloc(1);
    return call("hipStreamEndCapture");
}
hipError_t hipGraphInstantiate(void **e, void *, void **, char *, size_t) {
    *e = malloc(1);
    return call("hipGraphInstantiate");
}
hipError_t hipGraphDestroy(void *g) {
    free(g);
    return 0;
}
hipError_t hipGraphExecDestroy(void *e) {
    free(e);
    return 0;
}
hipError_t hipGraphLaunch(void *, void *) { return call("hipGraphLaunch"); }

hipError_t hipEventCreate(void **e) {
    *e = malloc(1);
    return 0;
}
hipError_t hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(void *e) {
    free(e);
    return 0;
}
hipError_t hipEventRecord(void *e, void *) {
    void *args[1] = {e};
    return call("hipEventRecord", args);
}
hipError_t hipEventSynchronize(void *) { return call("hipEventSynchronize"); }
hipError_t hipEventElapsedTime(float *ms, void *, void *) {
    *ms = 0;
    return call("hipEventElapsedTime");
}

}   /* extern "C" */
