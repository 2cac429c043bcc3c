// The library's host code over a HIP runtime of its own, which runs nothing:
// device memory is host memory that is never touched, a kernel launch is a line
// in the log, and two devices, streams and events are bookkeeping.  So what the
// host code asks of the runtime (on which device, in which order, how much) can
// be tested without a GPU.  The functions below take the place of the runtime's
// because the program's own symbols come first.
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <set>
#include <string>
#include <vector>

#include "nbx.h"

static int g_dev = 0;                        // current device
static size_t g_total = (size_t)288 << 30;   // memory of a device
static size_t g_used[2] = {0, 0}, g_peak = 0;
struct Alloc {
    size_t bytes;
    int dev;
};
static std::map<void *, Alloc> g_allocs;
static std::map<const void *, std::string> &names() {  // the library registers its kernels before this file's statics exist
    static auto *m = new std::map<const void *, std::string>;
    return *m;
}
struct FakeEvent {
    int dev, rec_dev;
    hipStream_t rec;
    bool pending;
};
static std::set<FakeEvent *> g_events;
static std::vector<std::string> g_log;
static bool g_fail_sync = false;
static hipError_t g_last = hipSuccess;

template <class... A>
static void note(const char *f, A... a) {
    char b[256];
    snprintf(b, sizeof(b), f, a...);
    g_log.push_back(b);
}
static void finish(bool (*which)(FakeEvent *, void *), void *arg) {
    for (FakeEvent *e : g_events)
        if (which(e, arg)) e->pending = false;
}
static hipError_t get(void **p, size_t n) {
    *p = nullptr;
    if (g_used[g_dev] + n > g_total) return hipErrorOutOfMemory;
    void *m = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    g_allocs[m] = {n, g_dev};
    g_used[g_dev] += n;
    if (g_used[g_dev] > g_peak) g_peak = g_used[g_dev];
    *p = m;
    return hipSuccess;
}
static hipError_t give(void *p) {
    if (!p) return hipSuccess;
    auto a = g_allocs.find(p);
    if (a == g_allocs.end()) return hipErrorInvalidValue;
    g_used[a->second.dev] -= a->second.bytes;
    munmap(p, a->second.bytes ? a->second.bytes : 1);
    g_allocs.erase(a);
    return hipSuccess;
}

extern "C" {
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *,
                           int *) {
    names()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
static dim3 p_grid, p_block;
static size_t p_shm;
static hipStream_t p_st;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shm, hipStream_t st) {
    p_grid = g;
    p_block = b;
    p_shm = shm;
    p_st = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shm, hipStream_t *st) {
    *g = p_grid;
    *b = p_block;
    *shm = p_shm;
    *st = p_st;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t st) {
    const uint64_t threads = (uint64_t)g.x * b.x;
    note("launch %s grid %u threads %llu stream %p", names()[f].c_str(), g.x, (unsigned long long)threads, (void *)st);
    if (threads >> 32) g_last = hipErrorInvalidConfiguration;
    return threads >> 32 ? hipErrorInvalidConfiguration : hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = g_dev;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    g_dev = d;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipDeviceTotalMem(size_t *v, hipDevice_t) {
    *v = g_total;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *v, const void *, int, size_t) {
    *v = 16;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) {
    note("device_sync dev %d", g_dev);
    if (g_fail_sync) return hipErrorStreamCaptureUnsupported;
    finish([](FakeEvent *e, void *) { return e->rec_dev == g_dev; }, nullptr);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t st) {
    finish([](FakeEvent *e, void *s) { return e->rec == (hipStream_t)s && e->rec_dev == g_dev; }, st);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t ev, unsigned) {
    FakeEvent *e = (FakeEvent *)ev;
    if (e->pending && e->rec != st) note("wait stream %p for stream %p", (void *)st, (void *)e->rec);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = hipStreamCaptureStatusNone;
    return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return g_dev; }
hipError_t hipEventCreateWithFlags(hipEvent_t *ev, unsigned) {
    FakeEvent *e = new FakeEvent{g_dev, -1, nullptr, false};
    g_events.insert(e);
    *ev = (hipEvent_t)e;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *ev) { return hipEventCreateWithFlags(ev, 0); }
hipError_t hipEventDestroy(hipEvent_t ev) {
    g_events.erase((FakeEvent *)ev);
    delete (FakeEvent *)ev;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t ev, hipStream_t st) {
    FakeEvent *e = (FakeEvent *)ev;
    e->rec = st;
    e->rec_dev = g_dev;
    e->pending = true;
    note("record dev %d stream %p", g_dev, (void *)st);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t ev) { return ((FakeEvent *)ev)->pending ? hipErrorNotReady : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t ev) {
    FakeEvent *e = (FakeEvent *)ev;
    if (e->pending) note("host waits for stream %p", (void *)e->rec);
    e->pending = false;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    const hipError_t e = get(p, n);
    note("malloc dev %d bytes %zu %s", g_dev, n, e == hipSuccess ? "ok" : "oom");
    return e;
}
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return get(p, n); }
hipError_t hipFree(void *p) {
    auto a = g_allocs.find(p);
    if (a != g_allocs.end()) note("free dev %d bytes %zu", a->second.dev, a->second.bytes);
    return give(p);
}
hipError_t hipFreeAsync(void *p, hipStream_t) { return give(p); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *at, const void *p) {
    auto a = g_allocs.find((void *)p);
    if (a == g_allocs.end()) return hipErrorInvalidValue;
    memset(at, 0, sizeof(*at));
    at->device = a->second.dev;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) {
    if (n <= 1 << 20 && k != hipMemcpyDeviceToDevice) memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *m = mmap(nullptr, (size_t)1 << 30, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    *p = m;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake"; }
}

static nbx_tree *tree(int64_t n, int form, hipStream_t st, bool vel = false) {
    nbx_params p;
    nbx_params_default(&p);
    p.form = form;
    nbx_tree *t = nullptr;
    // positions are only passed on
    const int rc = nbx_tree_create_dev(&p, (double *)64, vel ? (double *)64 : nullptr, nullptr, n, st, &t);
    if (rc) note("create failed %d", rc);
    return t;
}
static int32_t *const OUT = (int32_t *)64;

// One scenario, then the log from where it began to matter.
int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    const int64_t n = argc > 2 ? atoll(argv[2]) : 0;
    const int k = argc > 3 ? atoi(argv[3]) : 0;
    const hipStream_t A = (hipStream_t)0xA0, B = (hipStream_t)0xB0;
    size_t from = 0;
    if (what == "other_device" || what == "other_device_capturing") {
        // a tree of device 1, searched on a stream there, freed with device 0 current
        hipSetDevice(1);
        nbx_tree *t = tree(n, 0, A);
        nbx_density_dev(t, k, NBX_DENS_SYMMETRIC, 0, (double *)64, nullptr, A);
        nbx_knn_dev(t, k, NBX_KNN_NONPERIODIC, 0, OUT, nullptr, A);
        hipSetDevice(0);
        g_fail_sync = what != "other_device";
        from = g_log.size();
        nbx_tree_destroy(t);
        note("current dev %d", g_dev);
    } else if (what == "two_streams") {
        nbx_tree *t = tree(n, 0, A);
        nbx_knn_dev(t, k, NBX_KNN_NONPERIODIC, 0, OUT, nullptr, A);
        from = g_log.size();
        nbx_knn_dev(t, k, NBX_KNN_NONPERIODIC, 0, OUT, nullptr, B);
        note("%s", "again");
        nbx_knn_dev(t, k, NBX_KNN_NONPERIODIC, 0, OUT, nullptr, A);
        nbx_knn_dev(t, k, NBX_KNN_NONPERIODIC, 0, OUT, nullptr, B);
    } else if (what == "noalloc") {
        nbx_tree *t = tree(n, 0, A);
        from = g_log.size();
        const int rc = nbx_knn_density_noalloc(t, k, OUT, (double *)64, (double *)64, A);
        note("rc %d", rc);
    } else if (what == "rows" || what == "density") {
        nbx_tree *t = tree(n, argc > 4 ? atoi(argv[4]) : 0, A);
        from = g_log.size();
        const int rc = what == "rows" ? nbx_knn_dev(t, k, NBX_KNN_NONPERIODIC, 0, OUT, (double *)64, A)
                                      : nbx_density_dev(t, k, NBX_DENS_SYMMETRIC, 0, (double *)64, nullptr, A);
        note("rc %d", rc);
    } else if (what == "trim") {
        // a tree on each device, one search's block still in use
        for (int d = 0; d < 2; ++d) {
            hipSetDevice(d);
            nbx_tree_destroy(tree(n, 0, A));
        }
        nbx_tree *t = tree(n, 0, A);
        nbx_knn_dev(t, k, NBX_KNN_NONPERIODIC, 0, OUT, nullptr, A);
        const size_t before = g_used[0] + g_used[1];
        from = g_log.size();
        const int64_t got = nbx_trim_memory();
        note("trimmed %lld freed %zu left %zu again %lld", (long long)got, before - g_used[0] - g_used[1], g_used[0],
             (long long)nbx_trim_memory());
    } else if (what == "smooth") {
        // host arrays of this size are not copied
        nbx_tree *t = tree(n, 0, A, true);
        nbx_trim_memory();
        const size_t base = g_peak = g_used[0];
        from = g_log.size();
        double *const H = (double *)64;
        int rc = nbx_smooth_vel(t, k, nullptr, nullptr, H, nullptr);
        note("mean rc %d peak %zu", rc, g_peak - base);
        nbx_trim_memory();
        g_peak = base;
        rc = nbx_smooth_vel(t, k, nullptr, H, nullptr, H);
        note("disp rc %d peak %zu", rc, g_peak - base);
        nbx_trim_memory();
        g_peak = base;
        rc = nbx_smooth_vel_moments(t, k, nullptr, nullptr, H, H, H);
        note("moments rc %d peak %zu", rc, g_peak - base);
    } else if (what == "full") {
        // argv[4] bytes a particle are left beside the tree
        nbx_tree *t = tree(n, 0, A);
        nbx_trim_memory();
        g_total = g_used[0] + (size_t)atoll(argv[4]) * n + (1 << 20);
        from = g_log.size();
        int rc = nbx_knn_dev(t, k, NBX_KNN_NONPERIODIC, 0, OUT, (double *)64, A);
        note("rows rc %d", rc);
        rc = nbx_density_dev(t, k, NBX_DENS_SYMMETRIC, 0, (double *)64, nullptr, A);
        note("density rc %d", rc);
        rc = nbx_sph_density_fwd_tree_dev(t, k, 0, (double *)64, nullptr, A);
        note("spline rc %d", rc);
        nbx_tree_destroy(t);
        nbx_trim_memory();
        g_total = (size_t)288 << 30;
        t = tree(n, 0, A);
        nbx_trim_memory();
        g_total = g_used[0] + (size_t)(atoll(argv[4]) + 76 + 4 * k) * n + (1 << 20);
        rc = nbx_sph_density_adjoint_tree_dev(t, k, 0, (double *)64, (double *)64, (double *)64, A);
        note("adjoint rc %d", rc);
    } else if (what == "adjoint") {
        double *const D = (double *)4096;
        const int rc = nbx_sph_density_adjoint_ordered_dev(D, D, OUT, nullptr, n, k, D, D, D, D, A);
        note("rc %d", rc);
    } else if (what == "fof") {
        nbx_tree *t = tree(n, 0, A);
        from = g_log.size();
        int64_t ng = -1;
        const int rc = nbx_fof_dev(t, 0.1, 2, OUT, &ng, A);
        note("rc %d", rc);
    } else if (what == "build") {
        // n particles, form k, on a device of argv[4] GB
        if (argc > 4) g_total = (size_t)atoll(argv[4]) << 30;
        nbx_tree *t = tree(n, k, A);
        note("tree %d peak %zu held %zu", t != nullptr, g_peak, g_used[0]);
        from = g_log.size() - 1;
    } else {
        return 2;
    }
    for (size_t i = from; i < g_log.size(); ++i) puts(g_log[i].c_str());
    return 0;
}
