// The few runtime calls that transfer.hpp makes, on the CPU: a stream runs its work at once, an event is done as soon
// as it is recorded.  What a test wants to see or to go wrong is in fake.
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999, hipErrorNotReady = 600 };
struct FakeEvent {
    std::atomic<long> recorded{-1};  // number of the record
};
typedef FakeEvent* hipEvent_t;
typedef void* hipStream_t;
constexpr unsigned hipHostMallocDefault = 0x0, hipHostMallocCoherent = 0x40000000, hipEventDisableTiming = 0x2;

struct Fake {
    std::atomic<long> records{0};
    long fail_wait_of = -1;  // the wait for this record fails
    std::atomic<unsigned> host_flags{~0u}, host_allocs{0};  // flags that all host allocations had
};
inline Fake fake;

inline hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    fake.host_flags &= flags;
    fake.host_allocs++;
    *p = malloc(n);
    if (*p) memset(*p, 0xEE, n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = new FakeEvent, hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return e->recorded = fake.records++, hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    return fake.fail_wait_of >= 0 && e->recorded == fake.fail_wait_of ? hipErrorUnknown : hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) { return hipEventSynchronize(e); }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
