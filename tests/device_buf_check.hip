// device_buf_check.hip -- host checks of the device memory that the library's calls
// take (cusr_amd/csrc/device_buf.h, co_lib.hip) against a runtime of this file's own:
// an allocator of a limited size, whose errors stay until they are read
// (hipGetLastError), as the runtime's do; copies and launches that do nothing. Built
// and run by tests/test_device_buf.py with the check's name; prints "device buffers ok".
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>

#include "../cusr_amd/csrc/co_lib.hip"

using namespace cusr;

#define CHECK(c)                                        \
    do {                                                \
        if (!(c)) {                                     \
            printf("%s fails at line %d\n", #c, __LINE__); \
            exit(1);                                    \
        }                                               \
    } while (0)

namespace cusr {
#define LAUNCHER(name)                                                                          \
    hipError_t name##_0(int, unsigned, size_t, hipStream_t, const FitArgs &) { return hipSuccess; } \
    hipError_t name##_1(int, unsigned, size_t, hipStream_t, const FitArgs &) { return hipSuccess; } \
    hipError_t name##_2(int, unsigned, size_t, hipStream_t, const FitArgs &) { return hipSuccess; } \
    hipError_t name##_3(int, unsigned, size_t, hipStream_t, const FitArgs &) { return hipSuccess; }
LAUNCHER(launch_fit_f64_fwd)
LAUNCHER(launch_fit_f64_rev)
LAUNCHER(launch_fit_f32_fwd)
LAUNCHER(launch_fit_f32_rev)
LAUNCHER(launch_pass_f64_fwd)
LAUNCHER(launch_pass_f64_rev)
LAUNCHER(launch_pass_f32_fwd)
LAUNCHER(launch_pass_f32_rev)
}  // namespace cusr

static size_t g_size = 0, g_used = 0;
static hipError_t g_last = hipSuccess;
static std::map<void *, size_t> g_live;

extern "C" hipError_t hipMalloc(void **p, size_t n) {
    if (g_used + n > g_size) return g_last = hipErrorOutOfMemory;
    static uintptr_t next = 4096;
    *p = (void *)next;
    next += 4096;
    g_live[*p] = n;
    g_used += n;
    return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    CHECK(g_live.count(p));
    g_used -= g_live[p];
    g_live.erase(p);
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
extern "C" const char *hipGetErrorString(hipError_t) { return "out of memory"; }
extern "C" hipError_t hipSetDevice(int) { return hipSuccess; }
extern "C" hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
extern "C" hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = g_size - g_used;
    *t = g_size;
    return hipSuccess;
}
extern "C" hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    *v = 160 << 10;
    return hipSuccess;
}
extern "C" hipError_t hipGetSymbolAddress(void **p, const void *) {
    *p = (void *)64;
    return hipSuccess;
}
extern "C" hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = calloc(n, 1);
    return hipSuccess;
}
extern "C" hipError_t hipHostFree(void *p) {
    free(p);
    return hipSuccess;
}
extern "C" hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) {
    return hipSuccess;
}
extern "C" hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *) {
    a->type = hipMemoryTypeDevice;
    a->device = 0;
    return hipSuccess;
}
extern "C" hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *n, hipDeviceptr_t) {
    *base = nullptr;
    *n = (size_t)-1;
    return hipSuccess;
}
extern "C" hipError_t hipStreamCreateWithFlags(hipStream_t *, unsigned) { return hipSuccess; }
extern "C" hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
extern "C" hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
extern "C" hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
extern "C" hipError_t hipEventCreate(hipEvent_t *) { return hipSuccess; }
extern "C" hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipSuccess; }
extern "C" hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
extern "C" hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
extern "C" hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
extern "C" hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) {
    return hipSuccess;
}

// no device code is built or registered
extern "C" void **__hipRegisterFatBinary(const void *) { return nullptr; }
extern "C" void __hipUnregisterFatBinary(void **) {}
extern "C" void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, uint3 *,
                                      uint3 *, dim3 *, dim3 *, int *) {}
extern "C" void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

// A handle on a device of 1,000 MB with a data set of 100,000 points, and M
// expressions c0 sin(x0), each of one V column of 0.8 MB.
constexpr size_t kMB = 1000000;
struct Lib {
    void *handle = nullptr;
    CoOptions opt;
    PopHeader h = {};
    std::vector<int32_t> nt, ci, st;
    std::vector<float> nv;
    std::vector<TreeMeta> metas;
    std::vector<double> c, cf;
    Lib() {
        g_size = 1000 * kMB;
        CHECK(g_live.empty() && co_init(0, &handle) == CO_OK);
        co_options_default(&opt);
        opt.max_iter = 1;
        const double one = 0.0;
        CHECK(co_data_upload(handle, 100000, 1, &one, &one) == CO_OK);
    }
    ~Lib() {
        co_teardown(handle);
        CHECK(g_live.empty());
    }
    void population(int M) {
        nt.clear(), ci.clear(), nv.clear(), metas.clear();
        for (int m = 0; m < M; m++) {
            metas.push_back({4 * m, 4, m, 1});
            for (int t : {NODE_BFUNC, NODE_UFUNC, NODE_VAR, NODE_CONST}) nt.push_back(t);
            for (float v : {(float)OP_MUL, (float)OP_SIN, 0.0f, 0.0f}) nv.push_back(v);
            for (int k : {-1, -1, -1, 0}) ci.push_back(k);
        }
        h = {};
        h.magic = POP_MAGIC;
        h.version = POP_VERSION;
        h.M_prob = M;
        h.total_nodes = 4 * M;
        h.total_c = M;
        h.N = 100000;
        h.n_vars = 1;
        h.K_max = 1;
        h.max_stack = 2;
        c.assign(M, 0.0);
        cf.assign(M, 0.0);
        st.assign(M, 0);
    }
    int fit(int M) {
        population(M);
        return co_optimize_data(handle, &opt, &h, nt.data(), nv.data(), ci.data(), metas.data(),
                                c.data(), cf.data(), st.data(), nullptr, nullptr, nullptr);
    }
    int evaluate(int M) {
        population(M);
        double x = 0.0, y = 0.0;   // not read or written: no copy is made
        return co_eval_ex(handle, &h, nt.data(), nv.data(), ci.data(), metas.data(), c.data(), &x,
                          CO_PREC_FP64, &y);
    }
};

// What a call needs and the workspaces hold, the workspaces give back: an evaluation
// and both uploads of a data set, which fit the device only without them.
static void check_room() {
    const double v = 0.0;
    for (int call = 0; call < 3; call++) {
        Lib lib;
        CHECK(lib.fit(100) == CO_OK);
        CHECK(g_used > 100 * kMB && g_used < 110 * kMB);   // 100 MB of them workspace
        if (call == 0) CHECK(lib.evaluate(1150) == CO_OK);                                   // 920 MB
        if (call == 1) CHECK(co_data_upload(lib.handle, 38000000, 1, &v, &v) == CO_OK);      // 912 MB
        if (call == 2) CHECK(co_data_upload_device(lib.handle, 57000000, 1, &v, &v) == CO_OK);
        CHECK(g_used > 910 * kMB && g_used < 940 * kMB);
        // and a fit does without
        if (call == 0) CHECK(lib.fit(100) == CO_OK && g_used < 940 * kMB);
    }
}

// An allocation that fails leaves no error behind for the next launch's check, whether
// the workspaces make room for it or not.
static void check_error() {
    g_size = 1000;
    VWork v;
    v.max = 600;
    DevBuf b;
    v.set(0, 10, 5);   // 400 bytes and headroom
    CHECK(v.ptr[0]);
    CHECK(grow_needed(v, b, 900) == CO_OK && b.cap == 900 && !v.ptr[0]);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(grow_needed(v, b, 1100) == CO_ERR_OOM && b.cap == 0);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(grow(b, 1100) == CO_ERR_OOM);
    CHECK(hipGetLastError() == hipSuccess);
    CHECK(g_live.empty());
}

// A workspace and its headroom stay within the limit.
static void check_bound() {
    g_size = 100000;
    VWork v;
    v.max = 4000;
    for (int cols : {10, 100, 350, 400, 420, 500, 501, 3}) {
        for (int r = 0; r < kMaxRanges; r++) {
            v.set(r, cols, 1);
            CHECK((v.ptr[r] != nullptr) == (8 * cols <= 4000));
            if (v.ptr[r]) CHECK(v.buf[r].cap >= 8u * cols);
        }
        CHECK(g_used <= kMaxRanges * v.max);
    }
    CHECK(v.drop() && g_live.empty() && !v.drop());
}

int main(int argc, char **argv) {
    CHECK(argc == 2);
    if (!strcmp(argv[1], "error")) check_error();
    else if (!strcmp(argv[1], "room")) check_room();
    else if (!strcmp(argv[1], "bound")) check_bound();
    else CHECK(!"check's name");
    puts("device buffers ok");
    return 0;
}
