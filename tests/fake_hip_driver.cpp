// The engine's host side without a GPU, for tests/test_host_engine.py: this
// program defines the HIP calls that libgfc.so makes (its definitions come
// before libamdhip64's), with device memory in host memory and kernels that do
// nothing, so that error paths and launch decisions can be seen on the CPU.
//
// As in ROCm 7, an error stays the thread's last error until hipGetLastError
// reads it, whatever succeeds in between.
//
// Usage: fake_hip_driver <scenario> [numbers]; see main.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "gfc.h"

namespace {
struct Fake {
    std::mutex mu;
    std::map<const void *, std::string> kernels;
    std::vector<std::string> log;
    std::map<const char *, size_t> pinned;
    size_t most_pinned = ~(size_t)0;  // larger hipHostMalloc requests fail
    double sums = 1e3;                // what a reduction finds
    long sweeps_left = -1;            // sweep launches before one fails (< 0: none)
};
Fake &fake() {
    static Fake f;
    return f;
}
thread_local hipError_t last = hipSuccess;
thread_local bool no_memory = false;  // operator new fails on this thread
thread_local dim3 cfg_grid, cfg_block;

hipError_t err(hipError_t e) {
    last = e;
    return e;
}
// Memory for the driver itself.
struct Memory {
    const bool was = no_memory;
    Memory() { no_memory = false; }
    ~Memory() { no_memory = was; }
};
void note(const char *what, size_t n) {
    Memory m;
    std::lock_guard<std::mutex> lk(fake().mu);
    fake().log.push_back(std::string(what) + " " + std::to_string(n));
}
hipError_t alloc(void **p, size_t n) {
    *p = std::calloc(n ? n : 1, 1);
    return *p ? hipSuccess : err(hipErrorOutOfMemory);
}
}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
    fake().kernels[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) {
    cfg_grid = g;
    cfg_block = b;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shared, hipStream_t *s) {
    *g = cfg_grid;
    *b = cfg_block;
    *shared = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t) {
    Memory m;
    const std::string &name = fake().kernels[f];
    if (name.find("k_sweep") != std::string::npos && fake().sweeps_left >= 0 &&
        fake().sweeps_left-- == 0)
        return err(hipErrorLaunchFailure);
    note(("launch " + name + " " + std::to_string(g.x)).c_str(), b.x);
    if (name.find("k_reduce_final") != std::string::npos) {
        double *out = *static_cast<double **>(args[2]);
        for (int k = 0; k < 3; k++) out[k] = fake().sums;
    }
    if (name.find("k_sweep_slices") != std::string::npos)
        note(("sweeps " + std::to_string(*static_cast<int *>(args[5]))).c_str(),
             *static_cast<int *>(args[6]));
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) {
    return e == hipSuccess ? "no error" : e == hipErrorOutOfMemory ? "out of memory" : "error";
}
hipError_t hipGetLastError(void) {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = *t = (size_t)1 << 34;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { return alloc(p, 2u << 20); }
hipError_t hipMalloc(void **p, size_t n) { return alloc(p, n); }
hipError_t hipFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    if (n > fake().most_pinned) return err(hipErrorOutOfMemory);
    if (alloc(p, n) != hipSuccess) return hipErrorOutOfMemory;
    Memory m;
    fake().pinned[static_cast<char *>(*p)] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    fake().pinned.erase(static_cast<char *>(p));
    return hipFree(p);
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *ptr) {
    const char *p = static_cast<const char *>(ptr);
    *a = hipPointerAttribute_t{};
    a->type = hipMemoryTypeUnregistered;
    auto it = fake().pinned.upper_bound(p);
    if (it != fake().pinned.begin() && p < (--it)->first + it->second) a->type = hipMemoryTypeHost;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    note("copy", n);
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { return hipFree(s); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return hipFree(e); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 1;
    return hipSuccess;
}
}  // extern "C"

void *operator new(size_t n) {
    void *p = no_memory ? nullptr : std::malloc(n ? n : 1);
    if (p == nullptr) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

namespace {
// An FP64 configuration goes up and comes back, in pageable or pinned memory;
// prints the return codes, whether it came back as it was, and the message left
// behind.
int round_trip(gfc_ctx *c, gfc_geom g, bool pinned, bool starved) {
    const size_t n = (size_t)gfc_geom_volume(&g) * 72;
    void *m[2] = {nullptr, nullptr};
    for (void *&p : m) {
        if (pinned)
            (void)hipHostMalloc(&p, n * sizeof(double), 0);
        else
            p = std::calloc(n, sizeof(double));
    }
    double *U = static_cast<double *>(m[0]), *out = static_cast<double *>(m[1]);
    for (size_t k = 0; k < n; k++) U[k] = (double)k;
    gfc_job *j = nullptr;
    int rc = gfc_job_create(c, &g, GFC_PREC_FP64, &j);
    fake().log.clear();
    no_memory = starved;
    if (rc == GFC_OK) rc = gfc_job_upload_config(j, U, 8);
    const int up = rc;
    const int down = gfc_job_download_config(j, out);
    no_memory = false;
    std::printf("up %d down %d same %d message [%s]\n", up, down,
                (int)(std::memcmp(U, out, n * sizeof(double)) == 0), gfc_last_error());
    gfc_job_destroy(j);
    for (void *p : m) {
        if (pinned)
            (void)hipHostFree(p);
        else
            std::free(p);
    }
    return 0;
}
}  // namespace

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    auto arg = [&](int k) { return argc > k ? std::atol(argv[k]) : 0; };
    gfc_ctx *c = nullptr;
    if (gfc_ctx_create(0, &c) != GFC_OK) return 1;
    if (what == "no_ring") {
        // no_ring ns nt: pinned requests above 1 MiB fail
        fake().most_pinned = 1u << 20;
        round_trip(c, {(int)arg(2), (int)arg(3)}, false, false);
    } else if (what == "round_trip") {
        // round_trip ns nt pinned starved
        round_trip(c, {(int)arg(2), (int)arg(3)}, arg(4) != 0, arg(5) != 0);
    } else if (what == "fix") {
        // fix ns nt precision sweeps hits slice_group slice_lanes retire done:
        // the launch of half-sweep done + 1 fails if done is given; without
        // sweeps, the tolerance is one that the input meets
        gfc_geom g = {(int)arg(2), (int)arg(3)};
        gfc_params p;
        gfc_params_default(&p);
        p.tolerance = 1e-300;
        p.estimate_sweeps_to_gf_progress = 100000000;
        p.max_sweeps_to_fix = (unsigned)arg(5);
        p.hits = (unsigned)arg(6);
        if (arg(5) == 0) p.tolerance = 1e9;
        gfc_options o;
        gfc_options_default(&o);
        o.precision = (int)arg(4);
        o.slice_group = (int)arg(7);
        o.slice_lanes = (int)arg(8);
        o.retire_slices = (int)arg(9);
        gfc_job *j = nullptr;
        if (gfc_job_create(c, &g, o.precision, &j) != GFC_OK) return 1;
        fake().log.clear();
        gfc_report r{};
        fake().sweeps_left = argc > 10 ? arg(10) : -1;
        const int rc = gfc_job_fix(j, &p, &o, &r);
        fake().sweeps_left = -1;
        std::printf("fix %d sweeps %d message [%s]\n", rc, r.sweeps, gfc_last_error());
        gfc_job_destroy(j);
    } else if (what == "noalloc") {
        // noalloc offset: a configuration that many bytes behind a multiple of 16
        gfc_geom g = {4, 4};
        void *m = std::aligned_alloc(16, 4 * 4 * 4 * 4 * 576 + 16);
        double o[5];
        const int rc = gfc_config_observables_noalloc(
            c, &g, reinterpret_cast<double *>(static_cast<char *>(m) + arg(2)), o, o + 1, o + 2,
            o + 3, o + 4);
        std::printf("noalloc %d\n", rc);
        std::free(m);
    } else if (what == "trace") {
        // trace ns nt sweeps trace_len done: the launch of half-sweep done + 1
        // fails; 8 numbers behind the trace are looked at too
        gfc_geom g = {(int)arg(2), (int)arg(3)};
        gfc_params p;
        gfc_params_default(&p);
        p.tolerance = 1e-300;
        p.estimate_sweeps_to_gf_progress = 100000000;
        p.max_sweeps_to_fix = (unsigned)arg(4);
        gfc_job *j = nullptr;
        if (gfc_job_create(c, &g, GFC_PREC_FP64, &j) != GFC_OK) return 1;
        fake().log.clear();
        const int len = (int)arg(5);
        std::vector<double> tr(len + 8, -1.0);
        gfc_report r;
        fake().sweeps_left = arg(6);
        const int rc = gfc_job_fix_trace(j, &p, nullptr, &r, tr.data(), len);
        fake().sweeps_left = -1;
        int set = 0;
        while (set < (int)tr.size() && tr[set] > 0) set++;
        std::printf("trace %d set %d of %d\n", rc, set, len);
        gfc_job_destroy(j);
    } else {
        return 2;
    }
    for (const std::string &l : fake().log) std::printf("%s\n", l.c_str());
    gfc_ctx_destroy(c);
    return 0;
}
