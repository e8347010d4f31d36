// stage_main.cc -- the copies through pinned buffers (csrc/stage.h) against a
// runtime that this file makes up: copies run when their stream or an event
// behind them is waited for, and the n-th call of any kind can be made to fail.
// Prints OK and exits 0 when every check holds.
#include "../../tatsy-pppm_amd/csrc/stage.h"

#include <cstdio>
#include <cstdlib>
#include <functional>
#include <vector>

static int calls, fail_at = -1;          // calls made, the one that fails
static int buffers, events;              // alive
static std::vector<std::function<void()>> queue;  // the stream's work not yet done
static const char *pinned_lo, *pinned_hi;  // memory the runtime knows
static int copies, last_error;
static bool fails() { return calls++ == fail_at; }
static void drain() {
    for (auto& f : queue) f();
    queue.clear();
}

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (fails()) return hipErrorOutOfMemory;
    *p = std::malloc(n);
    buffers++;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    buffers--;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (fails()) return hipErrorOutOfMemory;
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    events++;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    if (!e) return hipErrorInvalidHandle;
    std::free(e);
    events--;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return !e ? hipErrorInvalidHandle : fails() ? hipErrorUnknown : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) {
    if (!e) return hipErrorInvalidHandle;
    if (fails()) return hipErrorUnknown;
    drain();
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    drain();
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (fails()) return hipErrorUnknown;
    copies++;
    queue.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    if (p < pinned_lo || p >= pinned_hi) return (hipError_t)(last_error = hipErrorInvalidValue);
    a->type = hipMemoryTypeHost;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = (hipError_t)last_error;
    last_error = hipSuccess;
    return e;
}
}

static int failures = 0;
static void expect(bool ok, const char* what, long at) {
    if (!ok) std::printf("FAIL: %s (%ld)\n", what, at), failures++;
}

int main() {
    std::vector<char> src(3 * STAGE_BYTES + 5), dst(src.size());
    for (size_t i = 0; i < src.size(); i++) src[i] = (char)(i * 2654435761u >> 13);
    // sizes about the ends of the buffers
    for (size_t n : {(size_t)0, (size_t)1, STAGE_BYTES - 1, STAGE_BYTES, STAGE_BYTES + 1, 2 * STAGE_BYTES, src.size()}) {
        HostStage st;
        std::fill(dst.begin(), dst.end(), 0);
        expect(st.copy_out(nullptr, dst.data(), src.data(), n) == hipSuccess, "copies", (long)n);
        expect(!std::memcmp(dst.data(), src.data(), n) && queue.empty(), "the bytes arrive", (long)n);
        expect(n == dst.size() || dst[n] == 0, "and no more", (long)n);
    }
    // every call fails once: the error is returned with nothing left in flight,
    // and the same object then copies
    for (int at = 0;; at++) {
        HostStage st;
        calls = 0;
        fail_at = at;
        const hipError_t e = st.copy_out(nullptr, dst.data(), src.data(), src.size());
        fail_at = -1;
        if (e == hipSuccess) break;
        expect(queue.empty(), "no copy is left on the stream", at);
        queue.clear();
        std::fill(dst.begin(), dst.end(), 0);
        expect(st.copy_out(nullptr, dst.data(), src.data(), src.size()) == hipSuccess, "works after a failure", at);
        expect(!std::memcmp(dst.data(), src.data(), src.size()), "with the right bytes", at);
    }
    // pinned memory: one copy, straight there, no buffers made
    pinned_lo = dst.data();
    pinned_hi = pinned_lo + dst.size();
    for (size_t n : {(size_t)1, STAGE_BYTES + 1, src.size()}) {
        HostStage st;
        copies = 0;
        std::fill(dst.begin(), dst.end(), 0);
        expect(st.copy_out(nullptr, dst.data(), src.data(), n) == hipSuccess, "copies to pinned memory", (long)n);
        expect(!std::memcmp(dst.data(), src.data(), n) && queue.empty(), "the bytes arrive there", (long)n);
        expect(copies == 1 && buffers == 0, "in one copy", copies);
    }
    expect(hipGetLastError() == hipSuccess, "no error is left behind", 0);
    expect(buffers == 0 && events == 0, "everything is given back", buffers + events);
    if (!failures) std::printf("OK\n");
    return failures != 0;
}
