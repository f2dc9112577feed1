// device_buf.h -- the library's device buffers: grown as needed and kept with the
// handle, and the workspaces of the V values, which a fit can do without.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/cusr_co.h"

namespace cusr {

constexpr int kMaxRanges = 2;   // launch ranges of one fit (the upload pipeline's two)

struct DevBuf {
    void *p = nullptr;
    size_t cap = 0;
};

static inline int grow(DevBuf &b, size_t bytes) {
    if (bytes == 0) bytes = 256;
    if (bytes <= b.cap) return CO_OK;
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
    hipError_t e = hipMalloc(&b.p, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();   // it would stay for the next launch's check
        fprintf(stderr, "[cusr_co] hipMalloc(%zu) failed: %s\n", bytes, hipGetErrorString(e));
        b.p = nullptr;
        return (e == hipErrorOutOfMemory) ? CO_ERR_OOM : CO_ERR_CUDA;
    }
    b.cap = bytes;
    return CO_OK;
}

// Workspaces of the V values (program.h), one per launch range, and where the
// resident population's lie: null where the range has none or they would not fit.
struct VWork {
    DevBuf buf[kMaxRanges];
    void *ptr[kMaxRanges] = {};
    size_t max = 0;   // bytes that each may take: an eighth of the device's memory

    // The workspaces given back (a fit then runs V in every pass); true if there
    // were any. hipFree waits for the device.
    bool drop() {
        bool any = false;
        for (int r = 0; r < kMaxRanges; ++r) {
            if (buf[r].p) {
                (void)hipFree(buf[r].p);
                any = true;
            }
            buf[r] = DevBuf();
            ptr[r] = nullptr;
        }
        return any;
    }

    // The workspace of range r for `cols` columns of N values of 8 bytes, grown with
    // a quarter of headroom (to max) and kept. ptr[r] stays null, and no error is
    // returned, where it would pass max or does not fit.
    void set(int r, int64_t cols, int N) {
        DevBuf &b = buf[r];
        const size_t bytes = sizeof(double) * (size_t)cols * (size_t)N;
        ptr[r] = nullptr;
        if (bytes == 0 || bytes > max) return;
        if (bytes > b.cap) {
            if (b.p) (void)hipFree(b.p);
            b = DevBuf();
            const size_t want = bytes + bytes / 4 < max ? bytes + bytes / 4 : max;
            if (hipMalloc(&b.p, want) != hipSuccess) {
                (void)hipGetLastError();
                b = DevBuf();
                return;
            }
            b.cap = want;
        }
        ptr[r] = b.p;
    }
};

// grow for what a call needs: out of memory, it takes the place of the V
// workspaces.
static inline int grow_needed(VWork &v, DevBuf &b, size_t bytes) {
    int rc = grow(b, bytes);
    if (rc == CO_ERR_OOM && v.drop()) rc = grow(b, bytes);
    return rc;
}

}  // namespace cusr
