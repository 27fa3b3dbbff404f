// The pinned slots of runtime.hpp (tsr_lists, tsr_staging) over a pretended device: work runs only when something
// waits for it, and a chosen hipEventRecord fails. Every queued read of a slot has to find the bytes that were in
// it when it was queued, and the memory has to outlive the reads.
#include <hip/hip_runtime.h>

#include "runtime.hpp"

#include <cstdio>
#include <cstdlib>
#include <deque>

struct Read { const uint8_t * src; uint8_t * dst; size_t bytes; uint8_t want; };
static std::deque<Read> queue;                                    // queued reads of pinned memory, oldest first
static uint64_t n_queued, n_done;
static uint64_t recorded[256];                                    // event: the reads queued when it was recorded
static int n_events, fail_in = -1, n_bad;
static bool freed;

static void run_until(uint64_t n) {
    while (n_done < n && !queue.empty()) {
        const Read r = queue.front();
        queue.pop_front();
        ++n_done;
        if (freed || r.src[0] != r.want || r.src[r.bytes - 1] != r.want) ++n_bad;
    }
}
static int enqueue(void * dst, const void * src, size_t bytes) {
    queue.push_back({ (const uint8_t *)src, (uint8_t *)dst, bytes, ((const uint8_t *)src)[0] });
    ++n_queued;
    return 0;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus * s) { *s = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { run_until(n_queued); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t * e, unsigned) { *e = (hipEvent_t)(uintptr_t)++n_events; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    if (fail_in >= 0 && fail_in-- == 0) return hipErrorUnknown;
    recorded[(uintptr_t)e] = n_queued;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { run_until(recorded[(uintptr_t)e]); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { run_until(n_queued); return hipSuccess; }
hipError_t hipMalloc(void ** p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipFree(void * p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void ** p, size_t n, unsigned) { *p = malloc(n); freed = false; return hipSuccess; }
hipError_t hipHostFree(void * p) { freed = true; run_until(n_queued); free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void * d, const void * s, size_t n, hipMemcpyKind, hipStream_t) { enqueue(d, s, n); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
int tsr::hip_err(hipError_t e, const char *) { return e == hipSuccess ? 0 : TSR_HIP_E_HIP; }
int tsr_launch_fetch(void * dst, const void * host, size_t bytes, hipStream_t) { return enqueue(dst, host, bytes); }

int main() {
    static uint8_t dst[64], src[64];
    constexpr size_t kList = tsr_lists::kCopyBytes + 1u;
    for (int lists = 0; lists < 2; ++lists)
        for (int fail = -1; fail < 70; ++fail) {                  // which hipEventRecord fails (-1: none)
            for (int calls : { 1, 5, 70, 140 }) {
                fail_in = fail;
                n_events = 0;
                tsr_lists l;
                tsr_staging st;
                if (l.acquire(tsr_lists::kCopyBytes) != nullptr || l.acquire(tsr_lists::kSlotBytes + 1u) != nullptr) return 3;
                for (int i = 0; i < calls; ++i) {
                    if (lists) {
                        uint8_t * slot = l.acquire(kList);
                        if (slot == nullptr) return 2;
                        memset(slot, i + 1, kList);
                        (void)l.send(dst, kList, nullptr);
                    } else {
                        memset(src, i + 1, sizeof src);
                        (void)st.copy(dst, src, sizeof src, nullptr);
                    }
                }
                l.release();
                st.release();
                run_until(n_queued);
                if (n_bad) {
                    printf("%s: %d of %d reads wrong with hipEventRecord %d failing\n", lists ? "lists" : "staging", n_bad, calls, fail);
                    return 1;
                }
            }
        }
    printf("no slot was written or given back under a read\n");
    return 0;
}
