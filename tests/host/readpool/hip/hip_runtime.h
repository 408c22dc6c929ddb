// The HIP calls that lq_readpool.h makes, for readpool_check.cpp: two devices, a
// current one per thread, streams and events that remember theirs, and counts of
// what is alive.
#pragma once
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdlib>

enum hipError_t { hipSuccess = 0, hipErrorInvalidHandle = 400 };
typedef int hipDevice_t;
struct ihipStream { int device; };
struct ihipEvent { int device; };
typedef ihipStream* hipStream_t;
typedef ihipEvent* hipEvent_t;
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };

inline thread_local int t_device = 0;
inline std::atomic<int> n_events{0}, n_host{0};

inline hipError_t hipGetDevice(int* d) { *d = t_device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { *d = s ? s->device : t_device; return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = malloc(n); n_host++; return hipSuccess; }
inline hipError_t hipHostFree(void* p) { free(p); n_host--; return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new ihipEvent{t_device}; n_events++; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; n_events--; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    int d = 0;
    (void)hipStreamGetDevice(s, &d);
    return e->device == d ? hipSuccess : hipErrorInvalidHandle;
}
