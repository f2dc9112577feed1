// device_buf_check.hip -- host checks of cusr_amd/csrc/device_buf.h against an
// allocator of this file's own, of a limited size, whose errors stay until they are
// read (hipGetLastError), as the runtime's do. Built and run by
// tests/test_device_buf.py with the check's name; prints "device buffers ok".
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>

#include "../cusr_amd/csrc/device_buf.h"

using namespace cusr;

#define CHECK(c)                                        \
    do {                                                \
        if (!(c)) {                                     \
            printf("%s fails at line %d\n", #c, __LINE__); \
            exit(1);                                    \
        }                                               \
    } while (0)

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

int main(int argc, char **argv) {
    CHECK(argc == 2);
    if (!strcmp(argv[1], "error")) check_error();
    else CHECK(!"check's name");
    puts("device buffers ok");
    return 0;
}
