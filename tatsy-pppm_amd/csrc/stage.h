// stage.h -- copies from the device to the caller's memory.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#define STAGE_BYTES ((size_t)1 << 20)

// Two pinned buffers, one copied out while the other fills: the runtime's own
// way to pageable memory pins the caller's pages, which costs more at every size
// (32 KB 28 -> 18 us, 0.4 MB 194 -> 48, 6 MB 0.50 -> 0.36 ms, 54 MB 5.3 -> 4.3 ms).
struct HostStage {
    char* buf = nullptr;
    hipEvent_t ev[2] = {};

    HostStage() = default;
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;
    ~HostStage() {
        if (buf) (void)hipHostFree(buf);
        for (auto& e : ev)
            if (e) (void)hipEventDestroy(e);
    }

    // Makes what is not there yet: a call after a failed one completes the set.
    hipError_t ready() {
        hipError_t e;
        for (auto& x : ev)
            if (!x && (e = hipEventCreateWithFlags(&x, hipEventDisableTiming)) != hipSuccess) {
                x = nullptr;
                return e;
            }
        if (!buf && (e = hipHostMalloc((void**)&buf, 2 * STAGE_BYTES, hipHostMallocDefault)) != hipSuccess) {
            buf = nullptr;
            return e;
        }
        return hipSuccess;
    }

    // Device memory src to dst, behind the work on s; complete on return, also
    // where it fails (then no copy is left on s).  Memory that the runtime knows
    // (pinned, managed, a device's) takes one copy straight there.
    hipError_t copy_out(hipStream_t s, void* dst, const void* src, size_t bytes) {
        hipError_t e;
        if (known(dst)) {
            if ((e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
            return hipStreamSynchronize(s);
        }
        if ((e = ready()) != hipSuccess) return e;
        if ((e = staged(s, (char*)dst, (const char*)src, bytes)) != hipSuccess) (void)hipStreamSynchronize(s);
        return e;
    }

private:
    static bool known(const void* p) {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();  // pageable memory is an error to some runtimes
            return false;
        }
        return a.type != hipMemoryTypeUnregistered;
    }
    hipError_t staged(hipStream_t s, char* dst, const char* src, size_t bytes) {
        hipError_t e;
        const size_t chunks = (bytes + STAGE_BYTES - 1) / STAGE_BYTES;
        for (size_t k = 0; k <= chunks; k++) {
            if (k < chunks) {
                const size_t at = k * STAGE_BYTES;
                if ((e = hipMemcpyAsync(buf + (k & 1) * STAGE_BYTES, src + at, std::min(STAGE_BYTES, bytes - at),
                                        hipMemcpyDeviceToHost, s)) != hipSuccess)
                    return e;
                if ((e = hipEventRecord(ev[k & 1], s)) != hipSuccess) return e;
            }
            if (k > 0) {
                const size_t at = (k - 1) * STAGE_BYTES;
                if ((e = hipEventSynchronize(ev[(k - 1) & 1])) != hipSuccess) return e;
                std::memcpy(dst + at, buf + ((k - 1) & 1) * STAGE_BYTES, std::min(STAGE_BYTES, bytes - at));
            }
        }
        return hipSuccess;
    }
};
